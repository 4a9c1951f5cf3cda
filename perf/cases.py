"""Performance cases: what a user of the engine has it do, through its public entry points.

Every case is a synthetic grid (``lightsim2grid_amd.gridgen``) of ``n`` buses, solved to a mismatch of
1e-8 pu (at most 10 Newton iterations, 30 fast-decoupled ones), with injections drawn from the seed as
the repository's time series draws them: every load times lognormal noise (sigma 0.05), around a
level, the dispatch following the total load. Kinds of work:

  pf      one power flow per call through a solver class (host arrays in, V out), from a flat start
  pf_dev  one power flow per call on arrays resident on the device
  ca      a contingency analysis as a whole: ContingencyAnalysisCPP.compute, compute_flows, both results
  n1      a batch of line outages on device arrays, warm-started from the base case ("order" lines each)
  ts      a time series as a whole: TimeSeriesCPP.compute_Vs, compute_flows, both results
  chains  a time series on device arrays, in chains of "length" warm-started steps
  dc      a batch of line outages with the DC solver, on device arrays
  fdpf    a time series with the fast-decoupled (XB) solver, one chain, on device arrays

Forms: "fp64" and "mixed" (FP32 factors, FP64 mismatch and update). The mixed form states its iteration
counts as those of the FP64 form within one, so its results are V and the statuses; the other forms
return their iteration counts as well. A row that did not converge has no result: its voltages are
zeroed after the call, as the batch classes do by themselves.
"""
import ctypes
import dataclasses
import functools
import math

import numpy as np
import torch

from lightsim2grid_amd import ContingencyAnalysisCPP, SolverType, TimeSeriesCPP, abi, gridgen, solver
from lightsim2grid_amd import lightsim2grid_amd_cpp as cpp

TOL = 1e-8


def listed():
    return [
        # the smallest call: one power flow of a 14-bus teaching grid in an environment's step loop
        {"name": "pf_14", "kind": "pf", "n": 14, "form": "fp64", "rows": 1, "level": 0.9},
        # the same on a 118-bus grid with the mixed form
        {"name": "pf_118_mixed", "kind": "pf", "n": 118, "form": "mixed", "rows": 1, "level": 0.9},
        # an operator's single power flow of a 2000-bus transmission grid
        {"name": "pf_2000", "kind": "pf", "n": 2000, "form": "fp64", "rows": 1, "level": 0.9},
        # a single power flow of the largest grid, data resident on the device
        {"name": "pf_10000", "kind": "pf_dev", "n": 10000, "form": "fp64", "rows": 1, "level": 0.9},
        # security analysis of a 118-bus grid: every line, islanding ones among them, with its flows
        {"name": "ca_118", "kind": "ca", "n": 118, "form": "fp64", "rows": 0, "level": 0.9},
        # N-2 screening of a regional grid of an odd size: pairs of lines
        {"name": "n2_613", "kind": "n1", "n": 613, "form": "fp64", "rows": 701, "order": 2, "level": 0.9},
        # the full N-1 sweep of a 2000-bus grid in both forms
        {"name": "n1_2000_mixed", "kind": "n1", "n": 2000, "form": "mixed", "rows": 2128, "order": 1, "level": 0.9},
        {"name": "n1_2000_fp64", "kind": "n1", "n": 2000, "form": "fp64", "rows": 2128, "order": 1, "level": 0.9},
        # N-1 of a 10000-bus grid, a part of its outages per batch
        {"name": "n1_10000_mixed", "kind": "n1", "n": 10000, "form": "mixed", "rows": 1500, "order": 1, "level": 0.9},
        # a year of hourly power flows of a 118-bus grid
        {"name": "ts_118", "kind": "ts", "n": 118, "form": "fp64", "rows": 8760, "length": 8760, "level": 0.9},
        # DC screening of every outage of a 2000-bus grid
        {"name": "dc_2000", "kind": "dc", "n": 2000, "form": "fp64", "rows": 2128, "order": 1, "level": 0.9},
        # a season of hourly fast-decoupled power flows of a 118-bus grid
        {"name": "fdpf_118", "kind": "fdpf", "n": 118, "form": "fp64", "rows": 2190, "length": 2190, "level": 0.9},
    ]


def draw(rng):
    def spread(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["pf", "pf", "pf_dev", "ca", "n1", "n1", "n1", "ts", "chains", "dc", "fdpf"])
    form = rng.choice(["fp64", "mixed"])
    c = {"kind": kind, "n": 0, "form": form, "rows": 1, "level": round(rng.uniform(0.8, 0.95), 3)}
    if kind in ("pf", "pf_dev"):
        c["n"] = spread(14, 10000)
    elif kind == "ca":
        c["n"], c["rows"] = spread(14, 400), 0
    elif kind in ("n1", "dc"):
        c["n"] = spread(30, 9000)
        c["rows"] = spread(12, max(13, min(2400, 5_000_000 // c["n"])))
        c["order"] = rng.choice([1, 1, 2])
    else:
        c["n"] = spread(14, 700)
        c["rows"] = spread(24, max(25, min(8760, 500_000 // c["n"])))
        c["length"] = spread(2, 48) if kind == "chains" else c["rows"]
    if kind in ("dc", "fdpf"):
        c["form"] = "fp64"
    if kind == "fdpf":  # the method's own range: it does not converge on the larger synthetic grids
        c["n"] = rng.choice([14, 118])
        c["rows"] = c["length"] = spread(24, 2100)
    return c


# --- grids and inputs --------------------------------------------------------------------------

@functools.lru_cache(maxsize=None)
def grid_of(n):
    """The repository's named grid of n buses, or one of the same generator and proportions."""
    name = "case%d_synth" % n
    if name in gridgen.CONFIGS:
        return gridgen.make(name)
    if n <= 60:  # small grids: a single slack bus at full load, as the 14- and 118-bus ones
        return gridgen.generate(n, n + max(3, n * 2 // 5), max(2, n * 3 // 10), seed=3)
    return gridgen.generate(n, n * 27 // 20, n // 4, seed=n, distributed_slack=True,
                            loading=0.25 * min(1.0, (2000.0 / n) ** 0.21))


@functools.lru_cache(maxsize=None)
def open_lines(n):
    """The lines whose outage leaves the grid in one piece."""
    return np.nonzero(~gridgen.bridges(grid_of(n)))[0]


@functools.lru_cache(maxsize=1)
def engine():
    return abi.Context(0)


def outages(case, rng):
    """Lists of lines taken out: all of a grid's (every `rows` of them), or pairs that keep it connected."""
    g, lines, rows = grid_of(case["n"]), open_lines(case["n"]), case["rows"]
    if case["order"] == 1:
        if rows >= len(lines):
            return [[int(lines[k % len(lines)])] for k in range(rows)]
        return [[int(k)] for k in np.sort(rng.choice(lines, rows, replace=False))]
    got = []
    while len(got) < rows:
        a, b = (int(x) for x in rng.choice(lines, 2, replace=False))
        if connected(g, (a, b)):
            got.append(sorted((a, b)))
    return got


def connected(g, out):
    """Whether the grid without these lines still is in one piece (union of both ends of each line)."""
    top = np.arange(g.n)
    keep = np.ones(g.nbr, bool)
    keep[list(out)] = False
    f, t = g.f[keep], g.t[keep]
    while True:
        low = top.copy()
        np.minimum.at(low, f, top[t])
        np.minimum.at(low, t, low[f])
        low = low[low]
        if np.array_equal(low, top):
            return not top.any()
        top = low


def injections(case, rng):
    """Sbus [rows or 1, n] of the case: noisy loads around the level, with the day's and year's cycles in a series."""
    g = grid_of(case["n"])
    rows = case["rows"] if case["kind"] in ("ts", "chains", "fdpf") else 1
    h = np.arange(rows)
    cycle = (1 + 0.25 * np.sin(2 * np.pi * h / 24)) * (1 + 0.15 * np.sin(2 * np.pi * h / 8760)) if rows > 1 else np.ones(1)
    scale = case["level"] * cycle[:, None] * rng.lognormal(0.0, 0.05, (rows, g.n))
    if rows > 1:  # the peak of both cycles stays within the level that the grid carries
        scale /= 1.25 * 1.15
    gen = (scale * g.load_p).sum(axis=1) / g.load_p.sum()
    return scale, gen, g.loading * (g.gen_p * gen[:, None] - (g.load_p + 1j * g.load_q) * scale)


def ybus_dc(g):
    """The DC matrix of the grid: 1/x stamps on the pattern of its Ybus."""
    y = 1.0 / g.x
    Y = g.ybus()
    Y.data[:] = 0.0
    for r, c, v in ((g.f, g.f, y), (g.t, g.t, y), (g.f, g.t, -y), (g.t, g.f, -y)):
        np.add.at(Y.data, positions(Y, r, c), v)
    return Y


def positions(Y, rows, cols):
    """Places of the entries (rows, cols) among the values of Y."""
    return np.array([Y.indptr[c] + np.searchsorted(Y.indices[Y.indptr[c]:Y.indptr[c + 1]], r) for r, c in zip(rows, cols)])


class Dev:
    """An array on the device as the engine's entry points take it."""

    def __init__(self, array):
        self.t = torch.as_tensor(array).cuda() if not torch.is_tensor(array) else array
        self.ptr = ctypes.c_void_p(self.t.data_ptr())


def pieces(case, seed):
    """The case's inputs from the seed alone, on the host."""
    rng = np.random.default_rng(seed)
    g = grid_of(case["n"])
    scale, gen, S = injections(case, rng)
    out = outages(case, rng) if case["kind"] in ("n1", "dc") else None
    return g, scale, gen, np.ascontiguousarray(S, np.complex128), out


def prepare(case, seed):
    kind, mixed = case["kind"], case["form"] == "mixed"
    g, scale, gen, S, out = pieces(case, seed)
    d = g.solver_inputs(sbus=S[0])
    s = {"case": case, "g": g}
    if kind == "pf":
        s["solver"] = solver.AMDGPUMixedSolver() if mixed else solver.AMDGPUSolver()
        s["args"] = (d["Ybus"], d["V0"], d["Sbus"], d["slack_ids"], d["slack_weights"], d["pv"], d["pq"], 10, TOL)
        return s
    if kind in ("ca", "ts"):
        load, bus = g.pq, np.r_[g.slack, g.pv]
        now = dataclasses.replace(g, gen_p=g.gen_p * gen[0], load_p=g.load_p * scale[0], load_q=g.load_q * scale[0])
        gm = gridgen.to_gridmodel(now)
        s["V0"] = g.v0()
        s["calc"] = (ContingencyAnalysisCPP if kind == "ca" else TimeSeriesCPP)(gm)
        s["calc"].change_solver(SolverType.AMDGPUMixed if mixed else SolverType.AMDGPU)
        if kind == "ca":
            s["calc"].add_all_n1()
        else:
            s["gen_p"] = np.ascontiguousarray(g.loading * g.gen_p[bus] * gen[:, None])
            s["load_p"] = np.ascontiguousarray(g.loading * g.load_p[load] * scale[:, load])
            s["load_q"] = np.ascontiguousarray(g.loading * g.load_q[load] * scale[:, load])
            s["sgen_p"] = np.zeros((case["rows"], 0))
        return s
    ctx = engine()
    Y = ybus_dc(g) if kind == "dc" else d["Ybus"]
    fdpf = None
    if kind == "fdpf":
        gm = gridgen.to_gridmodel(g)
        fdpf = (gm.debug_get_Bp_python(cpp.FDPFMethod.XB), gm.debug_get_Bpp_python(cpp.FDPFMethod.XB))
    gr = abi.Grid(ctx, Y, d["slack_ids"], d["slack_weights"], d["pv"], d["pq"], dc=kind == "dc", fdpf=fdpf)
    Yx = gr.ybus_values(Y)
    V0 = g.v0()
    if kind == "n1":  # warm start: the base case's own solution
        base = gr.solve(Yx, S[0], V0, 10, TOL)
        assert base["status"][0] == 0, "the base case does not converge"
        V0 = base["V"][0]
    rows = case["rows"]
    s["grid"], s["prec"] = gr, abi.FP32 if mixed else abi.FP64
    s["Y"], s["S"], s["V0"] = Dev(Yx), Dev(S), Dev(V0)
    s["V"] = Dev(torch.zeros((rows, g.n, 2), dtype=torch.float64, device="cuda"))
    s["it"], s["st"] = (Dev(torch.zeros(rows, dtype=torch.int32, device="cuda")) for _ in range(2))
    if out is not None:
        if kind == "dc":
            s["deltas"] = tuple(Dev(x) for x in dc_deltas(g, Y, out))
        else:
            s["deltas"] = tuple(Dev(x) for x in g.ybus_deltas(out))
    torch.cuda.synchronize()
    return s


def dc_deltas(g, Y, out):
    """The edits of the DC matrix for each list of lines, as Grid.ybus_deltas gives them for the AC one."""
    br = np.array([k for lines in out for k in lines])
    f, t, y = g.f[br], g.t[br], 1.0 / g.x[br]
    pos = np.stack([positions(Y, r, c) for r, c in ((f, f), (t, t), (f, t), (t, f))], axis=1)
    val = np.stack([y, y, -y, -y], axis=1)
    ptr = np.cumsum([0] + [4 * len(lines) for lines in out])
    return ptr.astype(np.int32), pos.reshape(-1).astype(np.int32), val.reshape(-1).astype(np.complex128)


def run(s):
    case, kind, mixed = s["case"], s["case"]["kind"], s["case"]["form"] == "mixed"
    if kind == "pf":
        ok = s["solver"].compute_pf(*s["args"])
        got = {"V": s["solver"].get_V(), "ok": bool(ok)}
        return got if mixed else {**got, "iters": int(s["solver"].get_nb_iter())}
    if kind == "ca":
        s["calc"].compute(s["V0"], 10, TOL)
        s["calc"].compute_flows()
        return {"V": s["calc"].get_voltages(), "amps": s["calc"].get_flows()}
    if kind == "ts":
        ok = s["calc"].compute_Vs(s["gen_p"], s["sgen_p"], s["load_p"], s["load_q"], s["V0"], 10, TOL)
        s["calc"].compute_flows()
        return {"V": s["calc"].get_voltages(), "amps": s["calc"].get_flows(), "ok": int(ok)}
    gr, rows = s["grid"], case["rows"]
    if kind in ("chains", "fdpf"):
        gr.solve_chains_device(s["Y"], 0, s["S"], s["V0"], 0, s["V"], rows, case["length"], s["it"], s["st"],
                               30 if kind == "fdpf" else 10, TOL, precision=s["prec"])
    else:
        gr.solve_device(s["Y"], 0, s["S"], 0, s["V0"], 0, s["V"], rows, s["it"], s["st"], 10, TOL,
                        precision=s["prec"], deltas=s.get("deltas"))
    if rows > 1:  # rows without a result; the engine's next call is on a stream of its own
        s["V"].t.masked_fill_((s["st"].t != 0)[:, None, None], 0.0)
        torch.cuda.current_stream().synchronize()
    got = {"V": s["V"].t, "status": s["st"].t}
    return got if mixed else {**got, "iters": s["it"].t}


def work(case):
    """Bytes: the injections, starts and edits read once, the results written once. Operations: per
    Newton iteration a sparse factorisation, two triangular solves and two products with Ybus, about
    20 log2(n) operations per bus on these grids; 4 iterations from a flat start, 3 from a warm one, 1
    for DC, and 13 (of a constant matrix, factored once) for the fast-decoupled method."""
    n, kind, rows = case["n"], case["kind"], case["rows"] or grid_of(case["n"]).nbr
    g = grid_of(n)
    series = kind in ("ts", "chains", "fdpf")
    read = 16.0 * (n + 2 * g.nbr) + 16.0 * n * (rows if series else 1) + 16.0 * n
    written = rows * (16.0 * n + 8.0)
    if kind in ("ca", "ts"):
        written += rows * 8.0 * g.nbr
    if kind in ("n1", "dc"):
        read += rows * case["order"] * 4 * 20.0
    per_it = 20.0 * n * math.log2(n)
    its = {"pf": 4, "pf_dev": 4, "dc": 0.5, "fdpf": 5}.get(kind, 3)
    return {"bytes": read + written, "flops": rows * its * per_it}


# --- the same results in plain torch, 64 bits ----------------------------------------------------

class Plain:
    """Newton's method on the power flow equations, batched over rows, with dense J (small grids) or
    with GMRES preconditioned by the base case's inverse J."""

    def __init__(self, g, S, out, dc=False):
        dev = "cuda" if torch.cuda.is_available() else "cpu"
        self.g, self.n, self.dev = g, g.n, dev
        t = lambda x, k=torch.float64: torch.as_tensor(np.ascontiguousarray(x), dtype=k, device=dev)  # noqa: E731
        self.f, self.t = t(g.f, torch.int64), t(g.t, torch.int64)
        yff, ytt, yft, ytf = g.branch_admittances()
        if dc:
            yff = ytt = 1.0 / g.x + 0j
            yft = ytf = -1.0 / g.x + 0j
        self.y = [t(v, torch.complex128) for v in (yff, yft, ytf, ytt)]
        ids = g.slack_ids
        self.pvpq = t(np.r_[ids[1:], g.pv_solver, g.pq], torch.int64)
        self.pq = t(g.pq, torch.int64)
        self.ref = int(ids[0])
        self.w = t(g.slack_weights())
        self.S = t(S, torch.complex128)
        rows = len(out) if out is not None else len(S)
        self.on = torch.ones((rows, g.nbr), dtype=torch.float64, device=dev)
        for k, lines in enumerate(out or ()):
            self.on[k, lines] = 0.0
        self.rows = rows

    def current(self, V, on):
        Vf, Vt = V[:, self.f] * on, V[:, self.t] * on
        I = torch.zeros_like(V)
        I.index_add_(1, self.f, self.y[0] * Vf + self.y[1] * Vt)
        I.index_add_(1, self.t, self.y[2] * Vf + self.y[3] * Vt)
        return I

    def pick(self, s):  # complex [.., n] -> the equations' rows
        return torch.cat([s[:, self.ref:self.ref + 1].real, s[:, self.pvpq].real, s[:, self.pq].imag], 1)

    def jx(self, V, I, on, x):
        k = len(self.pvpq)
        a = torch.zeros(V.shape, dtype=torch.float64, device=self.dev)
        m = a.clone()
        a[:, self.pvpq] = x[:, 1:1 + k]
        m[:, self.pq] = x[:, 1 + k:]
        dV = V * (1j * a + m / V.abs())
        return self.pick(dV * I.conj() + V * self.current(dV, on).conj() + x[:, :1] * self.w)

    def dense_j(self, V, on):
        n, k, B = self.n, len(self.pvpq), len(V)
        Y = torch.zeros((B, n, n), dtype=torch.complex128, device=self.dev)
        flat, at = Y.view(B, -1), lambda r, c: r * n + c  # noqa: E731
        for (r, c), y in zip(((self.f, self.f), (self.f, self.t), (self.t, self.f), (self.t, self.t)), self.y):
            flat.index_add_(1, at(r, c), y * on)
        I = (Y @ V[:, :, None])[:, :, 0]
        eye = torch.eye(n, device=self.dev)
        dA = 1j * V[:, :, None] * (I[:, None, :] * eye - Y * V[:, None, :]).conj()
        Vn = V / V.abs()
        dM = V[:, :, None] * (Y * Vn[:, None, :]).conj() + (I.conj() * Vn)[:, None, :] * eye
        J = torch.zeros((B, 1 + k + len(self.pq), 1 + k + len(self.pq)), dtype=torch.float64, device=self.dev)
        rowsP = torch.cat([torch.tensor([self.ref], device=self.dev), self.pvpq])
        J[:, :1 + k, 0] = self.w[rowsP]
        J[:, :1 + k, 1:1 + k] = dA[:, rowsP][:, :, self.pvpq].real
        J[:, :1 + k, 1 + k:] = dM[:, rowsP][:, :, self.pq].real
        J[:, 1 + k:, 1:1 + k] = dA[:, self.pq][:, :, self.pvpq].imag
        J[:, 1 + k:, 1 + k:] = dM[:, self.pq][:, :, self.pq].imag
        return J

    def newton(self, V0, max_iter=10):
        """(V, converged within max_iter) of every row; the converged ones polished to rounding."""
        small = self.n <= 60
        V = torch.as_tensor(V0, dtype=torch.complex128, device=self.dev).expand(self.rows, self.n).clone()
        sa = torch.zeros((self.rows, 1), dtype=torch.float64, device=self.dev)
        ok = torch.zeros(self.rows, dtype=torch.bool, device=self.dev)
        part = 128 if small else 2200
        inv = None if small else torch.linalg.inv(self.dense_j(V[:1], self.on[:1] * 0 + 1)[0])
        for a in range(0, self.rows, part):
            b = slice(a, min(self.rows, a + part))
            on, S = self.on[b], self.S if len(self.S) == 1 else self.S[b]
            v, z = V[b], sa[b]
            k = len(self.pvpq)
            for it in range(max_iter + 4):
                I = self.current(v, on)
                F = self.pick(v * I.conj() - S + z * self.w)
                if it <= max_iter:
                    ok[b] |= F.abs().amax(1) < TOL
                live = torch.isfinite(F).all(1) & (ok[b] | (it < max_iter))
                F = torch.where(live[:, None], F, torch.zeros_like(F))
                if small:
                    J = self.dense_j(v, on)
                    J[~live] = torch.eye(J.shape[1], dtype=torch.float64, device=self.dev)
                    x = torch.linalg.solve(J, F)
                else:
                    x = gmres(lambda u: self.jx(v, I, on, u), lambda u: u @ inv.T, F)
                z = z - x[:, :1]
                ang, mag = v.angle(), v.abs()
                ang[:, self.pvpq] -= x[:, 1:1 + k]
                mag[:, self.pq] -= x[:, 1 + k:]
                v = torch.polar(mag.abs(), torch.where(mag < 0, ang + math.pi, ang))
            V[b] = torch.where(ok[b][:, None], v, torch.zeros_like(v))
        return V, ok

    def linear(self):
        """Angles of the DC power flow, [rows, n], 0 at the reference."""
        k = self.pvpq
        P = self.S[:, k].real.expand(self.rows, len(k))
        full = torch.ones((1, self.g.nbr), dtype=torch.float64, device=self.dev)
        B = torch.zeros((self.n, self.n), dtype=torch.float64, device=self.dev).view(1, -1)
        for (r, c), y in zip(((self.f, self.f), (self.f, self.t), (self.t, self.f), (self.t, self.t)), self.y):
            B.index_add_(1, r * self.n + c, (y.real * full))
        inv = torch.linalg.inv(B.view(self.n, self.n)[k][:, k])

        def op(x):
            th = torch.zeros((len(x), self.n), dtype=torch.complex128, device=self.dev)
            th[:, k] = x.to(torch.complex128)
            return self.current(th, self.on)[:, k].real

        x = gmres(op, lambda u: u @ inv.T, P)
        th = torch.zeros((self.rows, self.n), dtype=torch.float64, device=self.dev)
        th[:, k] = x
        return th


def gmres(op, pre, b, m=12, restarts=4):
    """Batched restarted GMRES, right-preconditioned; op and pre act on [rows, N]."""
    x = torch.zeros_like(b)
    for _ in range(restarts):
        r = b - op(x) if _ else b
        beta = r.norm(dim=1, keepdim=True)
        safe = torch.where(beta > 0, beta, torch.ones_like(beta))
        Q, Z = [r / safe], []
        H = torch.zeros((len(b), m + 1, m), dtype=b.dtype, device=b.device)
        for j in range(m):
            Z.append(pre(Q[j]))
            u = op(Z[j])
            for _again in range(2):
                for i in range(j + 1):
                    h = (Q[i] * u).sum(1, keepdim=True)
                    H[:, i, j] += h[:, 0]
                    u = u - h * Q[i]
            h = u.norm(dim=1, keepdim=True)
            small = h < 1e-13
            H[:, j + 1, j] = torch.where(small, torch.zeros_like(h), h)[:, 0]
            Q.append(torch.where(small, torch.zeros_like(u), u / torch.where(small, torch.ones_like(h), h)))
        A = H.transpose(1, 2) @ H
        A = A + 1e-14 * torch.eye(m, dtype=b.dtype, device=b.device)
        y = torch.linalg.solve(A, H[:, 0, :, None] * beta[:, :, None])[:, :, 0]
        x = x + sum(y[:, j:j + 1] * Z[j] for j in range(m))
    return x


def exact(case, seed):
    kind, n = case["kind"], case["n"]
    if n > 2600:  # a dense inverse of this size takes too long
        return None
    g, scale, gen, S, out = pieces(case, seed)
    if kind == "ca":
        out = [[] if cut else [k] for k, cut in enumerate(gridgen.bridges(g))]
    p = Plain(g, S, out, dc=kind == "dc")
    if kind == "dc":
        V = torch.polar(torch.as_tensor(g.vset, device=p.dev).expand(p.rows, n), p.linear())
        ok = torch.ones(p.rows, dtype=torch.bool)
    else:
        V0 = g.v0()
        if kind in ("n1", "ca"):  # from the base case
            V0 = Plain(g, S, None).newton(V0)[0][0]
        V, ok = p.newton(V0)
        if kind == "ca":  # an outage that splits the grid is not solved
            ok &= torch.as_tensor(~gridgen.bridges(g), device=p.dev)
            V = torch.where(ok[:, None], V, torch.zeros_like(V))
    got = {"V": V.cpu().numpy()}
    if kind in ("n1", "dc", "pf_dev", "chains", "fdpf"):
        got["V"] = got["V"].view(np.float64).reshape(p.rows, n, 2)
    elif kind == "pf":
        got["V"] = got["V"][0]
    else:
        y = p.y
        with np.errstate(all="ignore"):
            Ef, Et = got["V"][:, g.f], got["V"][:, g.t]
            amps = np.abs(Ef * np.conj(y[0].cpu().numpy() * Ef + y[1].cpu().numpy() * Et)) / (math.sqrt(3.0) * np.abs(Ef))
        if kind == "ca":
            for k in np.nonzero(ok.cpu().numpy())[0]:
                amps[k, out[k]] = 0.0
        got["amps"] = amps
    return got
