"""Lanes per system of checkpoint launches of real particles: one lane where the batch keeps the lanes
busy for longer than its costliest system takes, else 8."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _belt(model, n, seed):
    from assist_amd import synthetic
    states = np.zeros((n, 1, 6))
    states[:, 0] = synthetic.main_belt(model, n, np.random.default_rng(seed))
    return states


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("n,shortest,longest,lanes", [(140001, 5.0, 5.0, 1), (70001, 2.0, 2.0, 1), (20000, 2.0, 2.0, 8),
                                                      (50000, 2.0, 300.0, 8)])
def test_lanes_follow_the_share_of_the_costliest_system(gpu, ephem, model, n, shortest, longest, lanes, precision):
    from assist_amd import batch
    states = _belt(model, n, n)
    t1 = np.geomspace(shortest, longest, n)
    t1[1::2] *= -1.0
    cfg = batch.BatchConfig.default(precision=precision)
    full = batch.integrate_checkpoint(ephem, 0.0, t1, states, config=cfg)
    assert (full.status == 0).all()
    assert full.stats.lanes_per_system == lanes
    # the snapshots carry the lanes: a paused batch goes on with them and ends with the same bits
    half = batch.integrate_checkpoint(ephem, 0.0, t1, states, config=cfg, t_pause=0.5 * t1)
    assert half.stats.lanes_per_system == lanes and (half.snapshots[:, 7] == lanes).all()
    done = batch.integrate_checkpoint(ephem, 0.0, t1, half.states, config=cfg, resume=half.snapshots)
    assert done.stats.lanes_per_system == lanes
    np.testing.assert_array_equal(done.states, full.states)
    np.testing.assert_array_equal(done.steps, full.steps)


def test_lanes_with_spans_that_are_no_numbers(gpu, ephem, model):
    """An infinite span and a NaN in the queue keep the 8-lane kernel and end by their status."""
    from assist_amd import batch
    n = 70001
    states = _belt(model, n, 3)
    t1 = np.full(n, 2.0)
    t1[5], t1[9] = np.inf, np.nan
    r = batch.integrate_checkpoint(ephem, 0.0, t1, states, config=batch.BatchConfig.default(max_steps=50))
    assert r.stats.lanes_per_system == 8
    assert (r.status[[5, 9]] != 0).all() and (np.delete(r.status, [5, 9]) == 0).all()


def test_vectors_and_overrides_keep_their_lanes(gpu, ephem, model):
    from assist_amd import batch, synthetic
    n = 70001
    states = np.zeros((n, 2, 6))
    states[:, :1] = _belt(model, n, 4)
    states[:, 1] = synthetic.variational_identity(n, 1)[:, 0]
    r = batch.integrate_checkpoint(ephem, 0.0, np.full(n, 1.0), states)
    assert r.stats.lanes_per_system == 8 and (r.status == 0).all()
    for lanes in (1, 8):
        r = batch.integrate_checkpoint(ephem, 0.0, np.full(n, 1.0), states[:, :1],
                                       config=batch.BatchConfig.default(lanes_per_system=lanes))
        assert r.stats.lanes_per_system == lanes
