"""The 16-lane integration kernel (assist_amd/csrc/row_kernel.hip), which launches without overrides
run, against the 8-lane kernel (lanes_per_system = 8): every operation on a system's data is the same,
so states, step and evaluation counts are equal bit for bit.  Sizes are the edges of its launch shapes
(one system per wave, four per wave, two waves per SIMD), vector counts those of its instances (the
real particle alone, up to 4 vectors, up to 8)."""
import numpy as np
import pytest

from conftest import population

pytestmark = pytest.mark.gpu


def _pair(ephem, t0, t1, states, params, precision=0, extras=None, **cfg):
    from assist_amd import batch
    rows = batch.integrate(ephem, t0, t1, states, params, extras=extras,
                           config=batch.BatchConfig.default(precision=precision, **cfg))
    groups = batch.integrate(ephem, t0, t1, states, params, extras=extras,
                             config=batch.BatchConfig.default(precision=precision, lanes_per_system=8, **cfg))
    assert rows.stats.lanes_per_system == 16 and groups.stats.lanes_per_system == 8
    return rows, groups


def _same(rows, groups):
    np.testing.assert_array_equal(rows.status, groups.status)
    np.testing.assert_array_equal(rows.steps, groups.steps)
    np.testing.assert_array_equal(rows.states, groups.states)
    assert (rows.stats.evals, rows.stats.rejected) == (groups.stats.evals, groups.stats.rejected)


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("n,n_var", [(1, 0), (1, 6), (5, 1), (67, 3), (67, 4), (67, 7), (1030, 6), (4100, 0), (5000, 7)])
def test_rows_equal_groups(gpu, ephem, model, n, n_var, precision):
    """Uneven spans in both directions (one of zero length), a third of the systems with a Marsden
    model."""
    from assist_amd import synthetic
    states, params, _ = population(model, n, 801 + n + n_var, n_var=n_var, ng_fraction=0.3)
    if n_var == 7:
        params[:, 7, 1] = 1e-12
    rng = np.random.default_rng(n)
    t0 = rng.uniform(-50.0, 50.0, n)
    t1 = t0 + synthetic.log_uniform_spans(n, rng, 2.0, 60.0 if n > 1000 else 250.0)
    if n > 2:
        t1[2] = t0[2]
    _same(*_pair(ephem, t0, t1, states, params, precision, min_dt=0.001))


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("forces", [0x7F, 0xFF, 0x13F, 0x05, 0x42, 0x38])
def test_rows_equal_groups_force_models(gpu, ephem, model, forces, precision):
    for n_var in (0, 6):
        states, params, _ = population(model, 40, 831, n_var=n_var, ng_fraction=0.3)
        # (a step limit: without the Sun's pull the mixed form's round-off drives some steps very small)
        _same(*_pair(ephem, 0.0, 90.0, states, params, precision, extras={"forces": forces}, min_dt=0.001, max_steps=200))
        # without Marsden parameters (kernels of their own for the default model)
        _same(*_pair(ephem, 0.0, -90.0, states, None, precision, extras={"forces": forces}, min_dt=0.001, max_steps=200))


@pytest.mark.parametrize("n_var", [0, 6])
def test_rows_rejections_failures_and_coverage(gpu, ephem, model, n_var):
    """First steps that are rejected, step limits, a non-finite state and the end of coverage."""
    states, _, _ = population(model, 50, 841, n_var=n_var, neo_fraction=0.0)
    r, g = _pair(ephem, 0.0, 600.0, states, None, dt_initial=500.0)
    assert r.stats.rejected >= 50
    _same(r, g)
    _same(*_pair(ephem, 0.0, 600.0, states, None, max_steps=9))
    _same(*_pair(ephem, 9950.0, np.linspace(9960.0, 10100.0, 50), states, None))
    bad = states.copy()
    bad[3, 0, 1] = np.nan
    bad[7, 0, 4] = np.inf
    r, g = _pair(ephem, 0.0, 40.0, bad, None)
    np.testing.assert_array_equal(r.status, g.status)
    ok = r.status == 0
    assert ok.sum() == 48
    np.testing.assert_array_equal(r.states[ok], g.states[ok])


@pytest.mark.parametrize("n_var", [0, 6])
def test_rows_dense_output(gpu, ephem, model, n_var):
    from assist_amd import batch
    n = 90
    states, _, _ = population(model, n, 851, n_var=n_var)
    rng = np.random.default_rng(851)
    outs = [np.sort(rng.uniform(0.0, 80.0, rng.integers(0, 9))) * (-1.0 if i % 2 else 1.0) for i in range(n)]
    outs = [o[::-1] if i % 2 else o for i, o in enumerate(outs)]
    outs = [np.sort(o) if not i % 2 else -np.sort(-o) for i, o in enumerate(outs)]
    rows = batch.integrate_dense(ephem, 0.0, outs, states)
    groups = batch.integrate_dense(ephem, 0.0, outs, states, config=batch.BatchConfig.default(lanes_per_system=8))
    assert rows.stats.lanes_per_system == 16 and (rows.status == 0).all()
    np.testing.assert_array_equal(rows.states, groups.states)
    for a, b in zip(rows.outputs, groups.outputs):
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("planets", ["asteroids of 13 coefficients", "no asteroids", "jpl binary"])
def test_rows_ephemeris_forms(gpu, model, tmp_path, planets):
    """Both lengths of the series in its ephemeris rounds, missing asteroid slots, and the records of a
    JPL binary file."""
    import assist_amd
    from assist_amd import synthetic
    pp, ap = synthetic.ensure_synthetic_ephemeris(0)
    if planets == "no asteroids":
        e = assist_amd.Ephem(pp)
    elif planets == "jpl binary":
        e = assist_amd.Ephem(synthetic.ensure_synthetic_ascii(0), ap)
    else:
        pp, ap = str(tmp_path / "p.bsp"), str(tmp_path / "a.bsp")
        synthetic.write_synthetic_ephemeris(pp, ap, 0, asteroid_record=(16.0, 13))
        e = assist_amd.Ephem(pp, ap)
    for precision in (0, 1):
        states, _, _ = population(model, 30, 861, n_var=2)
        _same(*_pair(e, -20.0, 200.0, states, None, precision, min_dt=0.001))


def test_rows_traces(gpu, ephem, model):
    """Step traces: the records of the 8-lane kernel, in another order."""
    from assist_amd import batch
    from assist_amd.learned import integrate_traced
    states, _, _ = population(model, 33, 871, n_var=2)
    got = []
    for lanes in (0, 8):
        rec = integrate_traced(ephem, np.zeros(33), np.full(33, 60.0), states, capacity=5000, skip=2,
                               config=batch.BatchConfig.default(lanes_per_system=lanes, min_dt=0.001))[0]
        got.append(rec[np.lexsort((rec[:, 1], rec[:, 0]))])
    np.testing.assert_array_equal(got[0], got[1])
