"""The one-lane kernel of real-only launches (lanes_per_system = 1) against the 16-lane kernel that small
batches run: the same integrator and force model with sums in another order.  Main-belt orbits over at
most 120 days, where a round-off of 1e-16 grows by less than 1e3 and the mixed form's stop leaves less
than 1e-11 of a position: 1 m (the 10-year bar of the parity tests) is wide for both, while a wrong
record, body or substep moves a position by kilometres."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
AU_M = 149597870700.0


def _both(ephem, t0, t1, states, params=None, **cfg):
    from assist_amd import batch
    lane = batch.integrate(ephem, t0, t1, states, params, config=batch.BatchConfig.default(lanes_per_system=1, **cfg))
    rows = batch.integrate(ephem, t0, t1, states, params, config=batch.BatchConfig.default(**cfg))
    assert lane.stats.lanes_per_system == 1 and rows.stats.lanes_per_system == 16
    return lane, rows


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("marsden", [False, True])
@pytest.mark.parametrize("n", [1, 63, 65, 1000])
def test_one_lane_against_rows(gpu, ephem, model, n, marsden, precision):
    """Both directions, start times over the records of every length (the lanes of a wave are in different
    ones, and steps cross their ends), and zero-length spans."""
    from assist_amd import synthetic
    rng = np.random.default_rng(910 + n)
    states = np.zeros((n, 1, 6))
    states[:, 0] = synthetic.main_belt(model, n, rng)
    params = None
    if marsden:
        params = np.zeros((n, 1, 3))
        params[:, 0] = synthetic.marsden_params(n, rng, 0.5)
    t0 = rng.uniform(-3000.0, 3000.0, n)
    t1 = t0 + rng.uniform(-120.0, 120.0, n)
    t1[:: 7] = t0[:: 7]
    lane, rows = _both(ephem, t0, t1, states, params, precision=precision)
    assert (lane.status == 0).all() and (rows.status == 0).all()
    np.testing.assert_array_equal(lane.states[:: 7], states[:: 7])
    assert (lane.steps[:: 7] == 0).all()
    d = np.linalg.norm(lane.states[:, 0, :3] - rows.states[:, 0, :3], axis=-1) * AU_M
    assert d.max() <= 1.0


def test_one_lane_statuses(gpu, ephem, model):
    """Coverage errors and the step limit end a system and leave the others of its wave alone."""
    from assist_amd import synthetic
    n = 130
    rng = np.random.default_rng(77)
    states = np.zeros((n, 1, 6))
    states[:, 0] = synthetic.main_belt(model, n, rng)
    t0, t1 = np.zeros(n), np.full(n, 100.0)
    t0[3::5], t1[3::5] = 9.0e4, 9.01e4   # outside the ephemeris from the start
    lane, rows = _both(ephem, t0, t1, states)
    np.testing.assert_array_equal(lane.status, rows.status)
    assert (lane.status[3::5] == 5).all() and (np.delete(lane.status, np.arange(3, n, 5)) == 0).all()
    lane, rows = _both(ephem, np.zeros(n), np.full(n, 400.0), states, max_steps=20)
    np.testing.assert_array_equal(lane.status, rows.status)
    assert (lane.status == -2).all() and (lane.steps == 20).all()


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("marsden", [False, True])
def test_last_systems_of_a_large_batch(gpu, ephem, model, marsden, precision):
    """In a batch of 131,072 systems or more every wave leaves its last systems to the 16-lane kernel: the
    same systems in batches below that stay on one lane throughout.  Lists of 128 and 129 systems a wave,
    zero-length spans and systems outside the ephemeris among them; twice the same bits."""
    from assist_amd import batch, synthetic
    n = 131072 + 65
    rng = np.random.default_rng(5)
    states = np.zeros((n, 1, 6))
    states[:, 0] = synthetic.main_belt(model, n, rng)
    params = None
    if marsden:
        params = np.zeros((n, 1, 3))
        params[:, 0] = synthetic.marsden_params(n, rng, 0.5)
    t0 = rng.uniform(-3000.0, 3000.0, n)
    t1 = t0 + rng.uniform(-60.0, 60.0, n)
    t1[::11] = t0[::11]
    t0[5::1001], t1[5::1001] = 9.0e4, 9.01e4
    cfg = batch.BatchConfig.default(lanes_per_system=1, precision=precision)
    whole = batch.integrate(ephem, t0, t1, states, params, config=cfg)
    again = batch.integrate(ephem, t0, t1, states, params, config=cfg)
    for k in ("states", "status", "steps"):
        np.testing.assert_array_equal(getattr(whole, k), getattr(again, k))
    h = n // 2
    parts = [batch.integrate(ephem, t0[s], t1[s], states[s], None if params is None else params[s], config=cfg)
             for s in (slice(0, h), slice(h, n))]
    np.testing.assert_array_equal(whole.status, np.concatenate([p.status for p in parts]))
    assert (whole.status[5::1001] == 5).all() and (whole.status == 5).sum() == len(t0[5::1001])
    ok = whole.status == 0
    d = np.linalg.norm(whole.states[:, 0, :3] - np.concatenate([p.states for p in parts])[:, 0, :3], axis=-1) * AU_M
    assert d[ok].max() <= 1.0
    # a step's length is the seventh root of its error estimate: round-off moves few step counts
    steps = np.concatenate([p.steps for p in parts])
    assert (np.abs(whole.steps - steps) <= 1).mean() > 0.999 and abs(whole.stats.steps - steps.sum()) < 1e-3 * steps.sum()


def test_large_batch_in_a_graph(gpu, ephem, model):
    """The captured launches of a large batch (counters, one-lane kernel, 16-lane kernel for the systems it
    leaves): every replay gives the eager launch's bits, with other work between them."""
    from assist_amd import batch, synthetic
    n = 131072 + 65
    rng = np.random.default_rng(8)
    states = np.zeros((n, 1, 6))
    states[:, 0] = synthetic.main_belt(model, n, rng)
    t0, t1 = rng.uniform(-2000.0, 2000.0, n), np.zeros(n)
    t1[:] = t0 + rng.uniform(-40.0, 40.0, n)
    d0, d1, first = batch.DeviceArray(t0), batch.DeviceArray(t1), batch.DeviceArray(states)
    st, status = batch.DeviceArray(states), batch.DeviceArray(np.zeros(n, np.int32))

    def run(**cfg):
        st.copy_from(first)
        batch.integrate_device(ephem, n, 0, d0, d1, st, None, status, None, None,
                               config=batch.BatchConfig.default(lanes_per_system=1, precision=1, **cfg))
        return st.download()

    eager = run()
    assert (status.download() == 0).all()
    for _ in range(3):
        np.testing.assert_array_equal(run(use_graph=1), eager)
        batch.synchronize()
        np.testing.assert_array_equal(run(), eager)
