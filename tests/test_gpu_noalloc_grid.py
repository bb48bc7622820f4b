"""The grid of the allocation-free entry point on 16 lanes per system: as large as the allocating one's
(its static scratch holds the records of every lane), with the same bits, and in about the same time."""
import ctypes as C
import time

import numpy as np
import pytest

from conftest import population

pytestmark = pytest.mark.gpu


def _runs(ephem, t0, t1, states, params, cfg, reps=1):
    """Final states, statuses and the best wall time of both entry points."""
    import assist_amd
    from assist_amd import batch
    n, nv = states.shape[:2]
    batch.get_particles(ephem, [0], [0.0])  # (the ephemeris must be resident)
    first, st = batch.DeviceArray(states), batch.DeviceArray(states)
    d0, d1, status = batch.DeviceArray(t0), batch.DeviceArray(t1), batch.DeviceArray(np.zeros(n, np.int32))
    pp = None if params is None else batch.DeviceArray(params)
    p = lambda x: None if x is None else C.c_void_p(x.ptr)  # noqa: E731
    args = [C.byref(ephem), None, C.byref(cfg), n, nv - 1, p(d0), p(d1), p(st), p(pp), p(status), None, None, None]
    lib, out = assist_amd.clibassist, []
    for call in (lambda: lib.assist_batch_integrate_device_noalloc(*args),
                 lambda: lib.assist_batch_integrate_device(*args, None)):
        best = np.inf
        for _ in range(reps):
            st.copy_from(first)
            batch.synchronize()
            begin = time.perf_counter()
            assert call() == 0
            best = min(best, time.perf_counter() - begin)
        out.append((st.download(), status.download(), best))
    return out


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("n,n_var,marsden", [(6200, 6, False), (6200, 7, True), (6200, 3, False), (13001, 0, True)])
def test_full_grid_equals_the_allocating_entry_point(gpu, ephem, model, n, n_var, marsden, precision):
    """More systems than the grid has rows (6,144, of four per wave)."""
    from assist_amd import batch
    states, params, _ = population(model, n, 91 + n_var, n_var=n_var, ng_fraction=0.3)
    rng = np.random.default_rng(n)
    t0 = rng.uniform(-50.0, 50.0, n)
    a, b = _runs(ephem, t0, t0 + rng.uniform(-30.0, 30.0, n), states, params if marsden else None,
                 batch.BatchConfig.default(precision=precision, min_dt=0.001))
    assert (a[1] == 0).all()
    np.testing.assert_array_equal(a[0], b[0])
    np.testing.assert_array_equal(a[1], b[1])


def test_as_fast_as_the_allocating_entry_point(gpu, ephem, model):
    """Equal spans of main-belt orbits, where the queue order that the entry point goes without matters
    little.  With two thirds of the grid it took 1.4 times as long."""
    from assist_amd import batch
    n = 65536
    states, _, _ = population(model, n, 97, n_var=6, neo_fraction=0.0)
    a, b = _runs(ephem, np.zeros(n), np.full(n, 60.0), states, None,
                 batch.BatchConfig.default(precision=batch.PRECISION_MIXED), reps=4)
    print("allocation-free %.2f ms, allocating %.2f ms" % (a[2] * 1e3, b[2] * 1e3))
    np.testing.assert_array_equal(a[0], b[0])
    assert a[2] < 1.25 * b[2]
