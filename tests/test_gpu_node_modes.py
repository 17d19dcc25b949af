"""The node kernel's instantiations: a plain run (eight changing compartments, constant coefficients) gives the same
bits alone and in a batch whose other runs bring optional features (the kernel with all of them), and the features
agree with the oracle where the kept contact row has edges.

Bar against the oracle: fixed steps to 1e-12 of a compartment's largest value over the run (a few hundred steps of
relative error 1.1e-16 on that scale, observed growth below ten).
"""
import numpy as np
import pytest

from memilio_amd import capi, synthetic
from memilio_amd.engine import Context
from memilio_amd.graphspec import E, INSC, ISYC
from tests import setups

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = Context()
    yield c
    c.close()


def _cfg(core):
    return {"ck": synthetic.ck_cfg(1e-8), "rkf45": setups.rkf45_cfg(1e-7, 1e-7, 1e-6, 1.0, dt=0.1),
            "fixed": synthetic.fixed_cfg(0.1),
            "euler": capi.sim_cfg(dt_node=0.1, integrator=capi.integrator_cfg(capi.INTEGRATOR_EULER, 0, 0, 0, 0))}[core]


def _featured(G, seed):
    sp = synthetic.graph(num_nodes=9, G=G, seed=seed, mean_degree=3.0)
    tot = sp.populations.sum(axis=(1, 2))
    sp.node_scalars[:, capi.P_TEST_AND_TRACE_CAPACITY] = 1e-4 * tot
    sp.node_scalars[:, capi.P_ICU_CAPACITY] = 1e-4 * tot
    sp.set_dampings([[(2.0, 0, 0, 0.4), (4.5, 1, 0, 0.3)]] * 9)
    sp.populations[:, :, INSC] = 5.0
    return sp


@pytest.mark.parametrize("core", ["ck", "rkf45", "fixed", "euler"])
@pytest.mark.parametrize("G", [1, 2, 3, 4, 5, 6, 7, 8])
def test_plain_run_alone_and_beside_features(ctx, G, core):
    plain = synthetic.graph(num_nodes=11, G=G, seed=70 + G, mean_degree=4.0)
    cfg = _cfg(core)
    alone, _ = ctx.ensemble_run([plain], [cfg], [9.0])
    both, _ = ctx.ensemble_run([plain, _featured(G, 80 + G)], [cfg, cfg], [9.0, 9.0])
    npis, _ = ctx.ensemble_run([plain, synthetic.with_npis(_featured(G, 80 + G))], [cfg, cfg], [9.0, 9.0])
    assert np.array_equal(alone[0], both[0])
    assert np.array_equal(alone[0], npis[0])


def _close(got, ref):
    scale = np.maximum(np.abs(ref).max(axis=0, keepdims=True), 1e-6)
    return float(np.max(np.abs(got - ref) / scale))


@pytest.mark.parametrize("times", [(3.0,), (3.0, 3.4), (0.0, 5.25, 5.25), (1.0, 2.0, 3.0, 11.0)])
def test_contact_rows_around_damping_days(ctx, oracle, times):
    """Dampings less than a day apart, at the start, at equal times, and outside of their days."""
    sp = synthetic.graph(num_nodes=10, G=3, seed=90, mean_degree=3.0)
    rng = np.random.default_rng(len(times))
    sp.contact_minimum = 0.1 * sp.contact_baseline
    sp.set_dampings([[(t, k % 2, k, rng.uniform(0.1, 0.5, (3, 3))) for k, t in enumerate(times)] if v % 3 else []
                     for v in range(10)])
    cfg = synthetic.fixed_cfg(0.1)
    out, _ = ctx.ensemble_run([sp], [cfg], [12.0])
    ref, _ = oracle.graph_run(sp, cfg, 12.0)
    assert _close(out[0], ref) < 1e-12


@pytest.mark.parametrize("compartment", [INSC, ISYC])
def test_confirmed_cases_at_the_start(ctx, oracle, compartment):
    """Initial confirmed cases in one group of one node: all ten compartments change."""
    sp = synthetic.graph(num_nodes=8, G=2, seed=91, mean_degree=3.0)
    sp.populations[5, 1, compartment] = sp.populations[5, 1, E]
    cfg = synthetic.fixed_cfg(0.1)
    out, _ = ctx.ensemble_run([sp], [cfg], [10.0])
    ref, _ = oracle.graph_run(sp, cfg, 10.0)
    assert _close(out[0], ref) < 1e-12
    assert out[0][1:, :, [compartment, 10 + compartment]].max() > 0
