"""Performance cases of the Graph-ODE engine, through its public entry points (memilio_amd/engine.py).

listed() holds twelve cases and draw() more of the same ranges; prepare() makes what a user's program has
in hand (sampled models, a resident batch, values on the device, a running serving loop), run() is one
pass, work() what a pass cannot do without and exact() the same results from plain torch / numpy in 64 bits.

Workloads come from memilio_amd/synthetic.py: graphs of 1..2000 nodes with 1..8 age groups, Poisson
out-degree up to 50, parameter studies around a base graph, horizons of weeks to half a year, adaptive
Cash-Karp and RKF45 at 1e-6..1e-10 and fixed steps of 0.1 day.
"""
import ctypes
import math

import numpy as np
import torch

from memilio_amd import capi, synthetic
from memilio_amd.engine import Batch, Context, GraphSim, Server
from memilio_amd.graphspec import E, ICR, INS, INSC, ISEV, ISY, ISYC, NC, R, D, S

PERCENTILES = (0.05, 0.25, 0.5, 0.75, 0.95)
ATTEMPTS_PER_DAY = {1e-6: 3.5, 1e-8: 8.0, 1e-10: 16.0}


def listed():
    return [
        # one calibrated model of six age groups over a season: the smallest call (osecir::simulate)
        {"name": "single_model", "kind": "single", "nodes": 1, "groups": 6, "days": 90, "core": "ck", "tol": 1e-10},
        # a handful of districts, one age split, the Runge-Kutta-Fehlberg core: a test-sized graph simulation
        {"name": "graph_24_rkf45", "kind": "graph", "nodes": 24, "groups": 3, "degree": 6, "days": 30, "core": "rkf45",
         "tol": 1e-8, "features": False},
        # all districts of a country, daily commuting, one run (make_mobility_sim + advance)
        {"name": "graph_400", "kind": "graph", "nodes": 400, "groups": 6, "degree": 50, "days": 100, "core": "ck",
         "tol": 1e-10, "features": False},
        # every model option at once: dampings, test-and-trace and ICU limits, commuter detection, a coefficient
        # per compartment on every edge; fixed step
        {"name": "graph_150_features", "kind": "graph", "nodes": 150, "groups": 4, "degree": 20, "days": 30,
         "core": "fixed", "tol": 0.0, "features": True},
        # a small study whose every trajectory is read back
        {"name": "study_48x150_daily", "kind": "study", "runs": 48, "nodes": 150, "groups": 5, "degree": 15,
         "days": 40, "core": "fixed", "tol": 0.0, "npis": False, "out": "daily"},
        # many samples of a small region without age groups, loose tolerance, summarised on the device
        {"name": "study_256x37", "kind": "study", "runs": 256, "nodes": 37, "groups": 1, "degree": 10, "days": 60,
         "core": "ck", "tol": 1e-6, "npis": False, "out": "stats"},
        # the parameter study of a country: the largest call
        {"name": "study_512x400", "kind": "study", "runs": 512, "nodes": 400, "groups": 6, "degree": 50, "days": 30,
         "core": "ck", "tol": 1e-10, "npis": False, "out": "stats"},
        # a study with dynamic NPIs on the contacts and on the commuting
        {"name": "study_64x100_npis", "kind": "study", "runs": 64, "nodes": 100, "groups": 6, "degree": 12,
         "days": 30, "core": "ck", "tol": 1e-8, "npis": True, "out": "stats"},
        # unrelated graphs of every size, age split, horizon and tolerance in one batch
        {"name": "uneven_48", "kind": "uneven", "graphs": 48, "max_nodes": 1000},
        # a burst of requests on the serving loop, submitted together and taken as they finish
        {"name": "serve_40", "kind": "serve", "graphs": 40, "max_nodes": 300},
        # percentiles of results that stay on the device (odd sizes)
        {"name": "percentiles_device", "kind": "device", "runs": 1000, "positions": 33333},
        # mean and percentiles of results that the program holds in host memory
        {"name": "statistics_host", "kind": "host", "runs": 101, "positions": 24400},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.499)))))))


def _core(rng):
    core = rng.choice(["ck", "ck", "ck", "rkf45", "fixed"])
    return core, (0.0 if core == "fixed" else rng.choice([1e-6, 1e-8, 1e-10]))


def draw(rng):
    kind = rng.choice(["single", "graph", "graph", "study", "study", "study", "uneven", "serve", "device", "host"])
    core, tol = _core(rng)
    if kind == "single":
        return {"kind": kind, "nodes": _log_int(rng, 1, 64), "groups": rng.randint(1, 8), "days": rng.randint(30, 180),
                "core": core, "tol": tol}
    if kind == "graph":
        return {"kind": kind, "nodes": _log_int(rng, 2, 2000), "groups": rng.randint(1, 8),
                "degree": rng.randint(2, 50), "days": rng.randint(20, 120), "core": core, "tol": tol,
                "features": rng.random() < 0.25}
    if kind == "study":
        nodes, groups, days = _log_int(rng, 5, 400), rng.randint(1, 8), rng.randint(10, 60)
        # at most the node-days and values of the largest listed study
        npis = rng.random() < 0.2
        runs = _log_int(rng, 8, max(8, min(128 if npis else 1024, 512 * 400 * 6 * 30 // (nodes * groups * days))))
        out = "daily" if runs <= 60 and runs * nodes * groups * days < 2_000_000 else "stats"
        return {"kind": kind, "runs": runs, "nodes": nodes, "groups": groups, "degree": rng.randint(2, 50),
                "days": days, "core": core, "tol": tol, "npis": npis, "out": out}
    if kind in ("uneven", "serve"):
        return {"kind": kind, "graphs": rng.randint(4, 48 if kind == "uneven" else 40),
                "max_nodes": _log_int(rng, 20, 1000 if kind == "uneven" else 300)}
    if kind == "device":
        runs = _log_int(rng, 5, 8000)
        return {"kind": kind, "runs": runs, "positions": _log_int(rng, 50, max(51, min(200_000, 40_000_000 // runs)))}
    runs = _log_int(rng, 5, 2000)
    return {"kind": kind, "runs": runs, "positions": _log_int(rng, 50, max(51, min(50_000, 4_000_000 // runs)))}


# ---------------------------------------------------------------------------------------------- inputs
_kept = {}


def _context():
    """The one context a program keeps for its simulations and studies."""
    if "ctx" not in _kept:
        _kept["ctx"] = Context()
    return _kept["ctx"]


def _server():
    """The one serving loop a program keeps, on a context of its own."""
    if "server" not in _kept:
        _kept["server_ctx"] = Context()
        _kept["server"] = Server(_kept["server_ctx"], hbm_budget_bytes=16 << 30, result_pool_bytes=1 << 30)
    return _kept["server"]


def _cfg(case):
    if case["core"] == "fixed":
        return synthetic.fixed_cfg(0.1)
    if case["core"] == "rkf45":
        return capi.sim_cfg(dt_node=0.1, integrator=capi.integrator_cfg(capi.INTEGRATOR_RKF45, case["tol"], case["tol"],
                                                                        1e-6, 1.0))
    return synthetic.ck_cfg(case["tol"])


def _models(case, seed):
    """Independent models (kind single)."""
    return synthetic.graph(case["nodes"], case["groups"], seed, mean_degree=0.0)


def _graph(case, seed):
    n, g = case["nodes"], case["groups"]
    spec = synthetic.graph(n, g, seed, mean_degree=float(min(case["degree"], n - 1)))
    if not case.get("features"):
        return spec
    rng = np.random.default_rng([seed, 7])
    tot = spec.populations.sum(axis=(1, 2))
    spec.node_scalars[:, capi.P_TEST_AND_TRACE_CAPACITY] = tot * rng.uniform(1e-5, 1e-3, n)
    spec.node_scalars[:, capi.P_ICU_CAPACITY] = tot * rng.uniform(1e-5, 1e-3, n)
    spec.node_scalars[:, capi.P_COMMUTER_NONDETECTION] = 0.6
    spec.node_scalars[:, capi.P_START_COMMUTER_DETECTION] = 2.0
    spec.node_scalars[:, capi.P_END_COMMUTER_DETECTION] = 15.0
    spec.contact_minimum = 0.2 * spec.contact_baseline
    spec.set_dampings([[(4.0, 0, 0, 0.5), (6.5, 1, 0, rng.uniform(0, 0.4, (g, g))), (12.0, 0, 0, 0.2)]
                       if v % 2 == 0 else [] for v in range(n)])
    spec.set_edges(spec.edge_start, spec.edge_end,
                   spec.edge_coeff_matrix() * rng.uniform(0.5, 1.0, (spec.num_edges, NC * g)))
    spec.populations[:, :, E:R] = spec.populations[:, :, E:E + 1] * rng.uniform(0.1, 1.0, (n, g, R - E))
    return spec


def _pool(case, seed):
    """Unrelated graphs: sizes, horizons and tolerances of the case, parameters and edges of the seed."""
    rng = np.random.default_rng([case["graphs"], case["max_nodes"]])
    specs, cfgs, tmax = [], [], []
    for k in range(case["graphs"]):
        n = max(1, min(case["max_nodes"], int(np.exp(rng.uniform(0.0, np.log(case["max_nodes"]))))))
        groups, days, tol = int(rng.integers(1, 9)), float(rng.integers(30, 181)), float(rng.choice([1e-6, 1e-8, 1e-10]))
        specs.append(synthetic.graph(n, groups, seed=seed * 64 + k, mean_degree=float(min(50, n - 1))))
        cfgs.append(synthetic.ck_cfg(tol))
        tmax.append(days)
    return specs, cfgs, tmax


def _study(case, seed):
    specs = synthetic.ensemble(_graph(case, seed), case["runs"], seed=seed + 1)
    if case["npis"]:
        for sp in specs:
            synthetic.with_edge_dampings(synthetic.with_npis(sp))
        for sp in specs[1:]:   # the samples of a study share the edges and their minimum
            sp.edge_coeff_minimum = specs[0].edge_coeff_minimum
    return specs


def _values(case, seed):
    """Results of a study: values of very different size, some compartments empty in every run."""
    gen = torch.Generator().manual_seed(seed)
    v = torch.randn(case["runs"], case["positions"], generator=gen, dtype=torch.float64).mul_(2.0).exp_()
    v[:, ::7] = 0.0
    return v


def prepare(case, seed):
    kind = case["kind"]
    state = {"case": dict(case)}
    if kind == "single":
        state.update(ctx=_context(), spec=_models(case, seed), cfg=_cfg(case))
    elif kind == "graph":
        state.update(ctx=_context(), spec=_graph(case, seed), cfg=_cfg(case))
    elif kind == "study":
        specs = _study(case, seed)
        state.update(batch=Batch(_context(), specs, [_cfg(case)] * len(specs), [float(case["days"])] * len(specs)))
    elif kind in ("uneven", "serve"):
        specs, cfgs, tmax = _pool(case, seed)
        if kind == "uneven":
            state.update(batch=Batch(_context(), specs, cfgs, tmax))
        else:
            state.update(server=_server(), requests=list(zip(specs, cfgs, tmax)))
    elif kind == "device":
        state.update(ctx=_context(), values=_values(case, seed).cuda(),
                     ps=np.array(PERCENTILES), out=torch.empty(len(PERCENTILES), case["positions"], dtype=torch.float64,
                                                               device="cuda"))
    else:
        state.update(ctx=_context(), values=_values(case, seed).numpy())
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "single":
        return state["ctx"].simulate_single(state["spec"], state["cfg"], float(case["days"]))
    if kind == "graph":
        sim = GraphSim(state["ctx"], state["spec"], state["cfg"], horizon=float(case["days"]))
        sim.advance(float(case["days"]))
        daily = sim.daily()
        sim.close()
        return daily
    if kind in ("study", "uneven"):
        batch = state["batch"]
        batch.reset()
        batch.run()
        if case.get("out") == "stats":
            return {"mean": batch.ensemble_mean(), "percentiles": batch.ensemble_percentiles(PERCENTILES)}
        return batch.read_daily()
    if kind == "serve":
        server = state["server"]
        tickets = [server.submit(*request) for request in state["requests"]]
        server.wait(tickets)
        return [server.take(ticket) for ticket in tickets]
    if kind == "device":
        ctx, stream = state["ctx"], torch.cuda.current_stream()
        ctx.check(ctx.lib.mgo_ensemble_percentiles_noalloc(
            ctx.ptr, ctypes.c_void_p(state["values"].data_ptr()), case["runs"], case["positions"],
            capi.dptr(state["ps"]), len(PERCENTILES), ctypes.c_void_p(state["out"].data_ptr()),
            ctypes.c_void_p(stream.cuda_stream)))
        return state["out"]
    return {"mean": state["ctx"].ensemble_mean_values(state["values"]),
            "percentiles": state["ctx"].ensemble_percentiles_values(state["values"], PERCENTILES)}


# ---------------------------------------------------------------------------------------------- work
def _sim_work(runs, nodes, groups, degree, days, attempts_per_day, out_values):
    """bytes: parameters and initial values in, results out; flops: step attempts (six right-hand sides of
    2 G^2 + 64 G + 7 and the stage sums of 540 G) and per edge and day the exchange (131 G)."""
    node_days = runs * nodes * days
    flops = node_days * (attempts_per_day * (6 * (2 * groups * groups + 64 * groups + 7) + 540 * groups)
                         + min(degree, nodes - 1) * 131 * groups)
    inputs = runs * nodes * (8 + 24 * groups + groups * groups) + 2 * nodes * min(degree, nodes - 1)
    return {"bytes": 8.0 * (inputs + out_values), "flops": float(flops)}


def work(case):
    kind = case["kind"]
    if kind in ("single", "graph", "study"):
        runs, n, g, days = case.get("runs", 1), case["nodes"], case["groups"], case["days"]
        per_run = (days + 1) * n * g * NC
        out = per_run * (1 + len(PERCENTILES)) if case.get("out") == "stats" else runs * per_run
        attempts = ATTEMPTS_PER_DAY.get(case["tol"], 10.0)
        return _sim_work(runs, n, g, case.get("degree", 0), days, attempts, out)
    if kind in ("uneven", "serve"):
        # log-uniform node counts, 1..8 groups, 30..180 days
        n = (case["max_nodes"] - 1) / math.log(case["max_nodes"])
        return _sim_work(case["graphs"], n, 4.5, 30, 105, 9.0, case["graphs"] * 106 * n * 45)
    values = case["runs"] * case["positions"]
    # every value read once; a selection compares each value with the wanted ranks at least once
    return {"bytes": 8.0 * (values + (1 + len(PERCENTILES)) * case["positions"]),
            "flops": float(values * math.ceil(math.log2(len(PERCENTILES) + 1)))}


# ---------------------------------------------------------------------------------------------- exact
# Cash-Karp 5th order with fixed fine steps: far more exact than any tolerance of the cases
_CK = (((), 0.0), ((1 / 5,), 1 / 5), ((3 / 40, 9 / 40), 3 / 10), ((3 / 10, -9 / 10, 6 / 5), 3 / 5),
       ((-11 / 54, 5 / 2, -70 / 27, 35 / 27), 1.0),
       ((1631 / 55296, 175 / 512, 575 / 13824, 44275 / 110592, 253 / 4096), 7 / 8))
_CK_B = (37 / 378, 0.0, 250 / 621, 125 / 594, 0.0, 512 / 1771)
_CK_ERR = (37 / 378 - 2825 / 27648, 0.0, 250 / 621 - 18575 / 48384, 125 / 594 - 13525 / 55296, -277 / 14336,
           512 / 1771 - 1 / 4)


class _Exact:
    """Plain torch simulation of runs that share one graph, scalar edge coefficients, no dampings or limits:
    y[run][node][group][compartment]."""

    def __init__(self, specs):
        dev = "cuda" if torch.cuda.is_available() else "cpu"
        stack = lambda name: torch.tensor(np.stack([getattr(s, name) for s in specs]), device=dev)  # noqa: E731
        a, sc = stack("age_params"), stack("node_scalars")
        p = lambda k: a[:, :, k, :]  # noqa: E731
        self.y = stack("populations")
        self.contact = stack("contact_baseline")
        self.start, self.season_k = sc[:, :, capi.P_START_DAY, None], sc[:, :, capi.P_SEASONALITY, None]
        self.tp = p(capi.A_TRANSMISSION_PROBABILITY_ON_CONTACT)
        self.rel = p(capi.A_RELATIVE_TRANSMISSION_NO_SYMPTOMS)
        self.risk = p(capi.A_RISK_OF_INFECTION_FROM_SYMPTOMATIC)
        t_e, t_ins, t_isy, t_isev, t_icr = (p(k) for k in range(5))
        rec, sev = p(capi.A_RECOVERED_PER_INFECTED_NO_SYMPTOMS), p(capi.A_SEVERE_PER_INFECTED_SYMPTOMS)
        crit, dsev = p(capi.A_CRITICAL_PER_SEVERE), p(capi.A_DEATHS_PER_SEVERE)
        dcr = p(capi.A_DEATHS_PER_CRITICAL)
        # linear flows (from, to, rate); the S -> E flow is added by rates()
        self.rates = [(E, INS, 1 / t_e), (INS, ISY, (1 - rec) / t_ins), (INS, R, rec / t_ins),
                      (INSC, ISYC, (1 - rec) / t_ins), (INSC, R, rec / t_ins), (ISY, ISEV, sev / t_isy),
                      (ISY, R, (1 - sev) / t_isy), (ISYC, ISEV, sev / t_isy), (ISYC, R, (1 - sev) / t_isy),
                      (ISEV, ICR, crit / t_isev), (ISEV, R, (1 - crit - dsev) / t_isev), (ISEV, D, dsev / t_isev),
                      (ICR, D, dcr / t_icr), (ICR, R, (1 - dcr) / t_icr)]
        spec = specs[0]
        order = np.lexsort((spec.edge_end, spec.edge_start))
        self.edges = list(zip(spec.edge_start[order].tolist(), spec.edge_end[order].tolist(),
                              spec.edge_coeffs[order].tolist()))
        n = spec.num_nodes
        self.coef = torch.zeros(n, n, dtype=torch.float64, device=dev)
        for s, d, c in self.edges:
            self.coef[s, d] = c

    def kappa(self, y, t):
        """S -> E rate per person."""
        alive = y[..., S] + y[..., E] + y[..., INS] + y[..., ISY] + y[..., ISEV] + y[..., ICR] + y[..., R]
        w = torch.where(alive < 1e-12, 0.0, (self.rel * y[..., INS] + self.risk * y[..., ISY]) / alive.clamp_min(1e-12))
        season = 1.0 + self.season_k * torch.sin(math.pi * ((self.start + t) / 182.5 + 0.5))
        return season * self.tp * (self.contact * w[..., None, :]).sum(-1)

    def slope(self, y, kappa, sel=slice(None)):
        out = torch.zeros_like(y)
        f = kappa * y[..., S]
        out[..., S] -= f
        out[..., E] += f
        for src, dst, rate in self.rates:
            f = rate[sel] * y[..., src]
            out[..., src] -= f
            out[..., dst] += f
        return out

    def advance(self, t, dt, steps):
        h = dt / steps
        for k in range(steps):
            ks = []
            for a, c in _CK:
                yt = self.y
                for w, kk in zip(a, ks):
                    yt = yt + (w * h) * kk
                ks.append(self.slope(yt, self.kappa(yt, t + k * h + c * h)))
            self.y = self.y + sum((b * h) * kk for b, kk in zip(_CK_B, ks) if b)

    def single(self, tol, days):
        """One model at a time with odeint's Cash-Karp controller (its daily values are interpolated between the
        steps that it chooses): [day][node][10 G]."""
        out, rates, whole = [], self.rates, (self.y, self.contact, self.start, self.season_k, self.tp, self.rel, self.risk)
        for v in range(whole[0].shape[1]):
            self.y, self.contact, self.start, self.season_k, self.tp, self.rel, self.risk = (x[:, v:v + 1] for x in whole)
            self.rates = [(src, dst, rate[:, v:v + 1]) for src, dst, rate in rates]
            y, t, dt, rows = self.y, 0.0, 0.1, [self.y.flatten()]
            while (days - t) / days > 1e-12:
                dt = min(dt, days - t)
                ks = []
                for a, c in _CK:
                    yt = y + sum((w * dt) * k for w, k in zip(a, ks))
                    ks.append(self.slope(yt, self.kappa(yt, t + c * dt)))
                err = sum((b * dt) * k for b, k in zip(_CK_ERR, ks)).abs()
                e = float((err / (tol + tol * (y.abs() + dt * ks[0].abs()))).max())
                if e > 1.0:
                    dt *= max(0.9 * e ** (-1.0 / 3.0), 0.2)
                    continue
                end = y + sum((b * dt) * k for b, k in zip(_CK_B, ks))
                while len(rows) <= days and len(rows) <= t + dt:
                    rows.append((y + (len(rows) - t) / dt * (end - y)).flatten())
                y, t = end, t + dt
                if e < 0.5:
                    dt *= 0.9 * max(5.0 ** -5, e) ** -0.2
            rows += [y.flatten()] * (days + 1 - len(rows))
            out.append(torch.stack(rows))
        return torch.stack(out, 1)

    def _mix(self, mat, v):
        """sum over nodes: out[r][j] = sum_i mat[i][j] v[r][i]."""
        r, n = v.shape[:2]
        flat = v.transpose(0, 1).reshape(n, -1).contiguous()
        return (mat.t().contiguous() @ flat).reshape(n, r, *v.shape[2:]).transpose(0, 1)

    def depart(self, t):
        self.gone = self.y.clone()
        self.gone[..., ISY] *= self.risk
        self.y = self.y + self._mix(self.coef, self.gone) - self.coef.sum(1)[None, :, None, None] * self.gone
        self.back = self.kappa(self.y, t)

    def come_back(self, h):
        """Every edge's travelers take one Euler step at their destination and return; a destination
        compartment that would fall below zero is filled from the group's largest one."""
        before = self.y
        arrived = self._mix(self.coef, self.gone)
        left = arrived + h * self.slope(arrived, self.back)
        # the travelers of all edges of a source, each with its destination's rates
        homes = torch.zeros_like(self.gone)
        homes += self.coef.sum(1)[None, :, None, None] * self.gone
        back_to = self.coef.t().contiguous()

        def flow(src, dst, rate):
            f = h * self._mix(back_to, rate[..., None])[..., 0] * self.gone[..., src]
            homes[..., src] -= f
            homes[..., dst] += f

        flow(S, E, self.back)
        for src, dst, rate in self.rates:
            flow(src, dst, rate)
        self.y = before - left + homes
        # a return in the edges' order where a compartment could have been short on the way
        low = ((before - left) < 0).flatten(1).any(1)
        if bool(low.any()):
            sel = torch.nonzero(low).flatten()
            self.y[sel] = self._in_order(before[sel], sel, h)

    def _in_order(self, y, sel, h):
        pick = lambda v: v[sel].cpu().numpy()  # noqa: E731
        y, gone, back = y.cpu().numpy(), pick(self.gone), pick(self.back)
        rates = [(src, dst, pick(rate)) for src, dst, rate in self.rates]
        for s, d, c in self.edges:
            m = c * gone[:, s]
            step = np.zeros_like(m)
            f = back[:, d] * m[..., S]
            step[..., S] -= f
            step[..., E] += f
            for src, dst, rate in rates:
                f = rate[:, d] * m[..., src]
                step[..., src] -= f
                step[..., dst] += f
            m = m + h * step
            left = y[:, d] - m
            if (left < 0).any():
                most = left.argmax(-1)[..., None]
                short = np.minimum(left, 0.0)
                np.put_along_axis(short, most, 0.0, -1)
                m += short
                np.put_along_axis(m, most, np.take_along_axis(m, most, -1) - short.sum(-1, keepdims=True), -1)
            y[:, s] += m
            y[:, d] -= m
        return torch.tensor(y, device=self.y.device)

    def daily(self, days, steps=8):
        out = [self.y.clone()]
        for day in range(days):
            t = float(day)
            self.advance(t, 0.5, steps)
            if self.edges:
                self.depart(t + 0.5)
            self.advance(t + 0.5, 0.5, steps)
            if self.edges:
                self.come_back(0.5)
            out.append(self.y.clone())
        return torch.stack(out, 1).flatten(3)   # [run][day][node][10 G]


def _statistics(v):
    """mean and percentiles over the first axis of v."""
    ranks = [int(v.shape[0] * p) for p in PERCENTILES]
    return {"mean": v.mean(0).cpu(), "percentiles": v.sort(0).values[ranks].cpu()}


def exact(case, seed):
    kind = case["kind"]
    if kind == "device":
        return _statistics(_values(case, seed))["percentiles"]
    if kind == "host":
        return _statistics(_values(case, seed))
    if kind not in ("single", "graph", "study") or case.get("features") or case.get("npis"):
        return None
    if kind == "single":
        if case["core"] != "ck" or case["nodes"] * case["days"] > 400:
            return None
        return _Exact([_models(case, seed)]).single(case["tol"], case["days"]).cpu()
    edges = case["nodes"] * min(case["degree"], case["nodes"] - 1)
    runs = case.get("runs", 1)
    if edges * case["days"] > 120_000 or runs * case["nodes"] * case["groups"] > 60_000:
        return None   # the edges' order is walked in Python
    if kind == "graph":
        return _Exact([_graph(case, seed)]).daily(case["days"])[0].cpu()
    daily = _Exact(_study(case, seed)).daily(case["days"])
    if case["out"] == "stats":
        return _statistics(daily)
    return [x.cpu() for x in daily]
