"""Downloads in chunks by several threads: sizes around the size from which they are used (8 MiB) and around a chunk
(1 MiB), every value in its place, bitwise (the mean of one run is the run itself), into pageable and pinned memory."""
import ctypes as C

import numpy as np
import pytest

from memilio_amd import capi, synthetic
from memilio_amd.engine import Batch, Context, Server

pytestmark = pytest.mark.gpu
MIB = 1 << 17   # doubles


@pytest.mark.parametrize("n", [1, 8 * MIB - 1, 8 * MIB, 8 * MIB + 1, 9 * MIB - 1, 9 * MIB + 1, 30 * MIB + 12345])
def test_large_results_arrive_whole(n):
    v = np.random.default_rng(n).normal(size=(1, n))
    with Context() as ctx:
        for _ in range(2):
            assert np.array_equal(ctx.ensemble_mean_values(v), v[0])


def test_runs_of_different_size_arrive_in_place():
    specs = [synthetic.graph(num_nodes=n, G=g, seed=n, mean_degree=3.0) for n, g in ((300, 6), (1, 1), (333, 8), (7, 2))]
    cfgs, tmaxs = [synthetic.ck_cfg(1e-6)] * 4, [60.0, 31.0, 45.0, 30.0]
    with Context() as ctx:
        batch = Batch(ctx, specs, cfgs, tmaxs)
        batch.run()
        whole = batch.read_daily()
        assert sum(x.nbytes for x in whole) > 8 << 20
        for k in range(4):
            assert np.array_equal(batch.read_daily(k, 1)[0], whole[k])
        batch.close()


@pytest.mark.parametrize("n,offset", [(8 * MIB - 1, 0), (8 * MIB, 3), (17 * MIB + 5, 1)])
def test_into_pinned_memory(n, offset):
    """Pinned results, also from within an allocation, take the plain copy."""
    v = np.random.default_rng(n).normal(size=n)
    with Context() as ctx:
        hip = C.CDLL("libamdhip64.so")
        p = C.c_void_p()
        assert hip.hipHostMalloc(C.byref(p), C.c_size_t((n + offset + 1) * 8), C.c_uint(0)) == 0
        out = np.frombuffer((C.c_double * (n + offset + 1)).from_address(p.value))
        out[:] = -1.0
        ctx.check(ctx.lib.mgo_ensemble_mean_values(ctx.ptr, capi.dptr(v), 1, n, capi.dptr(out[offset:offset + n])))
        assert np.array_equal(out[offset:offset + n], v)
        assert (out[:offset] == -1.0).all() and out[offset + n] == -1.0
        del out
        assert hip.hipHostFree(p) == 0


def test_served_results_beside_a_full_pool():
    """Results that find no room in the pinned pool, above and below the size of chunked downloads, are whole."""
    specs = [synthetic.graph(num_nodes=n, G=6, seed=n, mean_degree=3.0) for n in (300, 350, 40)]
    cfgs, tmaxs = [synthetic.ck_cfg(1e-6)] * 3, [60.0] * 3
    with Context() as ctx:
        want, _ = ctx.ensemble_run(specs, cfgs, tmaxs)
        assert want[0].nbytes > 8 << 20 > want[2].nbytes
        server = Server(ctx, result_pool_bytes=1 << 20)
        tickets = [server.submit(*r) for r in zip(specs, cfgs, tmaxs)]
        infos = server.wait(tickets)
        assert all(i.status == capi.OK for i in infos.values())
        for k, t in enumerate(tickets):
            assert np.array_equal(server.take(t), want[k])
        server.stop()
