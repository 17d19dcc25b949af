"""Percentile selection in registers against numpy's sort, bitwise: every list length and lane count of the kernels
(runs at and around 8, 16, ..., 4096 and above), positions around a block's, ties, empty compartments, infinities
and NaN (sorted last, as numpy does)."""
import numpy as np
import pytest

from memilio_amd.engine import Context

pytestmark = pytest.mark.gpu

PS = [0.001, 0.05, 0.25, 0.5, 0.75, 0.95, 0.999]
RUNS = [1, 2, 7, 8, 9, 16, 17, 32, 33, 63, 64, 65, 128, 129, 256, 257, 500, 512, 513, 1024, 1025, 2048, 2049, 4095,
        4096, 4097]


@pytest.fixture(scope="module")
def ctx():
    c = Context()
    yield c
    c.close()


def _values(runs, positions, seed):
    rng = np.random.default_rng([runs, positions, seed])
    v = rng.lognormal(0.0, 3.0, (runs, positions))
    v[:, 1::5] = np.round(v[:, 1::5])          # ties
    v[:, 2::7] = 0.0
    v[:, 3::11] *= -1.0
    v[rng.random((runs, positions)) < 0.01] = np.inf
    v[rng.random((runs, positions)) < 0.01] = -np.inf
    return v


@pytest.mark.parametrize("runs", RUNS)
def test_selection_equals_sorting(ctx, runs):
    for positions in (1, 3, 257, 1030):
        v = _values(runs, positions, 0)
        want = np.sort(v, axis=0)[[int(runs * p) for p in PS]]
        got = ctx.ensemble_percentiles_values(v, PS)
        assert np.array_equal(got, want), positions


@pytest.mark.parametrize("runs", [5, 64, 100, 700])
def test_nan_sorts_last(ctx, runs):
    v = _values(runs, 300, 1)
    v[np.random.default_rng(runs).random(v.shape) < 0.2] = np.nan
    v[:, 7] = np.nan
    want = np.sort(v, axis=0)[[int(runs * p) for p in PS]]
    assert np.array_equal(ctx.ensemble_percentiles_values(v, PS), want, equal_nan=True)
