"""Departures and returns where their closed form has edges: returns that must walk their edges (rates above one
per half day, negative travelers), susceptibles stepping below zero on the way (more than one infection per half
day), coefficient vectors, ICU limits, in-degrees around the walk's 64 / G edges at a time, more marked nodes than
a block lists at once, negative coefficients. Against the oracle, fixed steps.

Bar: every value to 1e-12 of its compartment's largest value over the run. A value is reached by at most a few
hundred edge and step operations of relative error 1.1e-16 on that scale, with observed growth below ten.
"""
import numpy as np
import pytest

from memilio_amd import capi, synthetic
from memilio_amd.engine import Context
from memilio_amd.graphspec import E, INS, S
from tests import setups

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = Context()
    yield c
    c.close()


def _check(ctx, oracle, spec, days, cfg=None, fixups=False):
    cfg = cfg or synthetic.fixed_cfg(0.1)
    out, info = ctx.ensemble_run([spec], [cfg], [float(days)])
    ref, st = oracle.graph_run(spec, cfg, float(days))
    if fixups:
        assert st.negative_fixups > 0
    if st.negative_fixups > 0:
        assert info.fixup_passes > 0
    scale = np.maximum(np.abs(ref).max(axis=0, keepdims=True), 1e-6)
    assert float(np.max(np.abs(out[0] - ref) / scale)) < 1e-12
    return info


@pytest.mark.parametrize("G", [1, 2, 3, 5, 6, 8])
def test_in_degrees_around_a_walk_step(ctx, oracle, G):
    """Node k of the graph has k in-edges, 0 .. 64 / G + 2 of them; heavy commuting, so that returns fall short."""
    n = 64 // G + 3
    sp = synthetic.graph(num_nodes=n, G=G, seed=40 + G, mean_degree=1.0)
    start, end = zip(*[(s, d) for d in range(n) for s in [x for x in range(n) if x != d][:d]])
    tot = np.bincount(start, minlength=n)
    sp.set_edges(np.array(start), np.array(end), 0.95 / np.maximum(tot, 1)[list(start)])
    sp.age_params[:, capi.A_RISK_OF_INFECTION_FROM_SYMPTOMATIC, :] = 0.05
    sp.populations[:, :, E] *= np.random.default_rng(G).uniform(1, 30, (n, G))
    _check(ctx, oracle, sp, 12)


def test_rates_above_one_per_half_day(ctx, oracle):
    """Stay times below the graph step: the Euler step of the travelers overshoots."""
    sp = setups.fixup_graph(seed=6, n=20, G=3)
    sp.age_params[::2, capi.A_TIME_INFECTED_NO_SYMPTOMS, :] = 0.4
    _check(ctx, oracle, sp, 10, synthetic.fixed_cfg(0.05))


@pytest.mark.parametrize("n,G", [(70, 1), (20, 3), (24, 8)])
@pytest.mark.parametrize("stay", [capi.A_TIME_EXPOSED, capi.A_TIME_INFECTED_NO_SYMPTOMS,
                                  capi.A_TIME_INFECTED_SYMPTOMS, capi.A_TIME_INFECTED_SEVERE,
                                  capi.A_TIME_INFECTED_CRITICAL])
def test_each_rate_above_one_per_half_day(ctx, oracle, stay, n, G):
    """One steep rate in every other node: its compartment's travelers turn negative at such destinations."""
    sp = setups.fixup_graph(seed=7, n=n, G=G, outflow=0.8)
    sp.age_params[::2, stay, :] = 0.3
    _check(ctx, oracle, sp, 8, synthetic.fixed_cfg(0.05))


@pytest.mark.parametrize("n,G", [(1, 1), (70, 1), (20, 3), (12, 8)])
def test_negative_coefficients(ctx, oracle, n, G):
    """Some edges carry travelers against their direction: every return walks its edges from the start."""
    sp = synthetic.graph(num_nodes=n + 1, G=G, seed=52, mean_degree=min(5.0, n))
    c = sp.edge_coeffs.copy()
    c[::3] *= -0.1
    c[1 % c.size] = abs(c[1 % c.size])
    sp.set_edges(sp.edge_start, sp.edge_end, c)
    _check(ctx, oracle, sp, 6)


@pytest.mark.parametrize("G", [1, 4])
def test_more_than_one_infection_per_half_day(ctx, oracle, G):
    """Force of infection above 1 / h: the returning susceptibles step below zero; the closed form still holds."""
    sp = synthetic.graph(num_nodes=18, G=G, seed=50, mean_degree=6.0)
    sp.contact_baseline *= 60.0 / G
    sp.populations[:, :, INS] = 0.3 * sp.populations[:, :, S]
    _check(ctx, oracle, sp, 6, synthetic.fixed_cfg(0.02))


@pytest.mark.parametrize("n,G", [(12, 3), (1100, 1)])
def test_negative_travelers(ctx, oracle, n, G):
    """A negative compartment in one node: every node of the run walks its edges (1100 nodes: more than one list)."""
    sp = synthetic.graph(num_nodes=n, G=G, seed=51, mean_degree=4.0)
    sp.populations[3, 0, INS] = -50.0
    info = _check(ctx, oracle, sp, 3)
    assert info.fixup_passes > 0


@pytest.mark.parametrize("icu", [False, True])
@pytest.mark.parametrize("dampings", [False, True])
def test_coefficient_vectors(ctx, oracle, icu, dampings):
    """One coefficient per compartment, some zero (compartments that do not travel); ICU limits; damped coefficients."""
    G = 3
    sp = setups.fixup_graph(seed=4, n=24, G=G)
    rng = np.random.default_rng(8)
    cv = sp.edge_coeff_matrix() * rng.uniform(0.5, 1.0, (sp.num_edges, 10 * G))
    cv.reshape(-1, G, 10)[:, :, 6:8] = 0.0
    sp.set_edges(sp.edge_start, sp.edge_end, cv)
    if icu:
        sp.node_scalars[::2, capi.P_ICU_CAPACITY] = 1e-4 * sp.populations[::2].sum(axis=(1, 2))
    if dampings:
        synthetic.with_edge_dampings(sp, thresholds=())
    _check(ctx, oracle, sp, 15)


@pytest.mark.parametrize("G", [2, 7])
def test_uniform_coefficients_with_icu_and_dampings(ctx, oracle, G):
    sp = setups.fixup_graph(seed=5, n=25, G=G)
    sp.node_scalars[1::2, capi.P_ICU_CAPACITY] = 1e-4 * sp.populations[1::2].sum(axis=(1, 2))
    synthetic.with_edge_dampings(sp, thresholds=())
    _check(ctx, oracle, sp, 15)


def test_fixups_settle_and_replay(ctx, oracle):
    """The fix-up graph: chains of fix-ups over several passes, and the same run resolved sequentially."""
    sp = setups.fixup_graph()
    _check(ctx, oracle, sp, 20, fixups=True)
    with Context(flags=capi.CTX_SEQUENTIAL_FIXUP) as seq:
        info = _check(seq, oracle, sp, 20, fixups=True)
        assert info.exact_replays > 0


@pytest.mark.parametrize("G", [1, 3, 6])
def test_edges_of_a_node_to_itself(ctx, oracle, G):
    """The first, a middle and the last of a node's edges lead back to it; also resolved sequentially."""
    n = 26
    sp = setups.fixup_graph(seed=12, n=n, G=G)
    loops = np.array([0, 7, 8, n - 1])
    start = np.concatenate([sp.edge_start, loops])
    c = np.concatenate([sp.edge_coeffs, [0.05, 0.02, 0.09, 0.05]])
    c *= 0.98 / np.bincount(start, weights=c)[start]
    sp.set_edges(start, np.concatenate([sp.edge_end, loops]), c)
    _check(ctx, oracle, sp, 6, fixups=True)
    with Context(flags=capi.CTX_SEQUENTIAL_FIXUP) as seq:
        _check(seq, oracle, sp, 6, fixups=True)


@pytest.mark.parametrize("G", [1, 2, 6, 8])
def test_replay_of_many_edges(ctx, oracle, G):
    """Out-degrees around the replay's 64 / G edges at a time, from 0 to 64 / G + 2."""
    most = 64 // G + 2
    n = max(40, most + 1)
    sp = setups.fixup_graph(seed=12, n=n, G=G)
    start, end = np.array([(s, (s + 1 + d) % n) for s in range(n) for d in range(s % (most + 1))]).T
    sp.set_edges(start, end, 0.98 / np.bincount(start)[start])
    with Context(flags=capi.CTX_SEQUENTIAL_FIXUP) as seq:
        info = _check(seq, oracle, sp, 6, fixups=True)
        assert info.exact_replays > 0


@pytest.mark.parametrize("n,G,runs", [(9, 8, 3), (70, 1, 40), (300, 3, 257), (1500, 1, 2), (1600, 1, 3)])
def test_shares_of_a_pass(ctx, oracle, n, G, runs):
    """A pass's nodes are shared out to 256 / runs blocks of eight wavefronts, at most one per node: the same bits
    alone (up to 64 blocks), beside one other run, in a large batch (one block). 1600 nodes: two launches."""
    sp = setups.fixup_graph(seed=9, n=n, G=G)
    _check(ctx, oracle, sp, 4, fixups=n > 9)
    alone, info = ctx.ensemble_run([sp], [synthetic.fixed_cfg(0.1)], [4.0])
    out, both = ctx.ensemble_run([sp] * runs, [synthetic.fixed_cfg(0.1)] * runs, [4.0] * runs)
    assert all(np.array_equal(o, alone[0]) for o in out)
    assert both.fixup_passes == runs * info.fixup_passes
