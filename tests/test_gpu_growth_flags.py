"""The growth flag of a row (pfgpu_ctx_last_flags) says that a pivot of its own factorisations lost its value to
cancellation. A workgroup of several instances walks on until its last one is done: the flags of the rows that are
done before must not depend on it, so they equal those of one instance per workgroup."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _say(*a):
    print("[gpu-case]", *a, flush=True)
    sys.stdout.flush()


# values in LDS, with V laid over them, and spilled
@pytest.mark.parametrize("n,G", [(60, 2), (60, 8), (118, 4), (400, 4), (900, 2), (900, 8)])
@pytest.mark.parametrize("prec", [0, 2])
def test_growth_flags_are_a_rows_own(gpu_ctx, n, G, prec):
    from lightsim2grid_amd import abi, gridgen
    _say("growth flags", n, G, prec)
    g = gridgen.make("case118_synth") if n == 118 else gridgen.generate(n, n + n // 2, n // 4, 3, loading=0.3)
    d = g.solver_inputs()
    gr = abi.Grid(gpu_ctx, d["Ybus"], d["slack_ids"], d["slack_weights"], d["pv"], d["pq"])
    Yx = gr.ybus_values(d["Ybus"])
    base = gr.solve(Yx, d["Sbus"], d["V0"], 10, 1e-8)
    assert base["status"][0] == 0
    # rows from close to the solution (one iteration) to far from it, in turn
    rng = np.random.default_rng(n)
    rows = 24
    V0 = np.repeat(base["V"], rows, axis=0)
    for i in range(rows):
        V0[i] *= 1 + (0.0, 1e-4, 0.05, 0.3)[i % 4] * (rng.standard_normal(g.n) + 1j * rng.standard_normal(g.n)) / 3
    r1 = gr.solve(Yx, d["Sbus"], V0, 10, 1e-8, precision=prec, instances_per_wg=1)
    f1 = gpu_ctx.last_flags(rows) & abi.FLAG_GROWTH
    rG = gr.solve(Yx, d["Sbus"], V0, 10, 1e-8, precision=prec, instances_per_wg=G)
    fG = gpu_ctx.last_flags(rows) & abi.FLAG_GROWTH
    assert rG["stats"]["instances_per_wg"] == G and len(set(r1["iters"].tolist())) > 2
    # of the rows that converge, hence end before the diverging ones of their workgroup (whose own path, and with it
    # their flag, is set by the rounding of the last sums, which the launch shape orders)
    done = r1["status"] == 0
    assert np.array_equal(done, rG["status"] == 0) and done[0::4].all() and done[1::4].all() and not done[3::4].all()
    assert np.array_equal(f1[done], fG[done])
    assert not f1[0::4].any() and not f1[1::4].any()
