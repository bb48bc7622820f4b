"""Systems that the one-lane kernel leaves to the 16-lane kernel at the end of a large real-only batch,
where steps are rejected and where the step limit ends them: counts, statuses and times as on 8 lanes,
states to round-off.  Main-belt orbits over at most 300 days, where a round-off of 1e-16 of 3 au grows by
less than 1e3 (0.05 m): 1 m (the bar of the parity tests) holds it, and a lost system, count or correction
moves a position by kilometres."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
AU_M = 149597870700.0
N = 131072 + 65


def _runs(ephem, model, seed, **cfg):
    from assist_amd import batch, synthetic
    rng = np.random.default_rng(seed)
    states = np.zeros((N, 1, 6))
    states[:, 0] = synthetic.main_belt(model, N, rng)
    t1 = rng.uniform(200.0, 300.0, N) * np.where(np.arange(N) % 2, -1.0, 1.0)
    out = [batch.integrate(ephem, 0.0, t1, states, config=batch.BatchConfig.default(lanes_per_system=lanes, **cfg))
           for lanes in (0, 8)]
    assert out[0].stats.lanes_per_system == 1 and out[1].stats.lanes_per_system == 8
    return out


@pytest.mark.parametrize("precision", [0, 1])
def test_rejected_steps_across_the_hand_over(gpu, ephem, model, precision):
    one, groups = _runs(ephem, model, 5 + precision, precision=precision, dt_initial=250.0)
    assert (one.status == 0).all() and (groups.status == 0).all()
    assert groups.stats.rejected > N // 2  # (the first trial step is too long for most)
    assert abs(one.stats.rejected - groups.stats.rejected) <= 1e-3 * groups.stats.rejected
    assert (np.abs(one.steps - groups.steps) <= 1).mean() > 0.999
    d = np.linalg.norm(one.states[:, 0, :3] - groups.states[:, 0, :3], axis=-1) * AU_M
    print("rejections %d and %d, max %.3g m" % (one.stats.rejected, groups.stats.rejected, d.max()))
    assert d.max() <= 1.0


@pytest.mark.parametrize("precision", [0, 1])
def test_step_limit_across_the_hand_over(gpu, ephem, model, precision):
    """Nine steps from a trial step of 0.001 days grow fourfold each at most, to tens of days."""
    one, groups = _runs(ephem, model, 9, precision=precision, max_steps=9)
    assert (one.status == -2).all() and (groups.status == -2).all()
    assert (one.steps == 9).all() and (groups.steps == 9).all()
