"""A paused and resumed run against plain integration of the same batch, which runs other kernels: the
16-lane kernel by default and the one-lane kernel for lanes_per_system = 1."""
import numpy as np
import pytest

from conftest import AU_M, population

pytestmark = pytest.mark.gpu


def _resumed(ephem, t0, t1, states, params, lanes, precision, at=0.4, **kw):
    from assist_amd import batch
    cfg = batch.BatchConfig.default(lanes_per_system=lanes, precision=precision, **kw)
    half = batch.integrate_checkpoint(ephem, t0, t1, states, params, config=cfg, t_pause=t0 + at * (t1 - t0))
    assert (half.status == batch.SYSTEM_PAUSED).all()
    done = batch.integrate_checkpoint(ephem, t0, t1, half.states, params, resume=half.snapshots,
                                      config=batch.BatchConfig.default(precision=precision, **kw))
    assert (done.status == 0).all()
    return done, batch.integrate(ephem, t0, t1, states, params, config=cfg)


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("n_var,lanes", [(0, 0), (0, 8), (3, 0), (6, 0), (7, 8), (0, 2), (2, 4)])
def test_resumed_equals_plain(gpu, ephem, model, n_var, lanes, precision):
    """Bit for bit in double precision, and for the real particle in the mixed form.  There the kernels with
    and without the checkpoint features round a few FP32 partials differently (2^-24 of terms that are
    1e-8 of the Sun's pull: 1e-15 of a vector an evaluation, 1e-12 with a growth of 10 over 100 steps)."""
    states, params, _ = population(model, 70, 401 + n_var, n_var=n_var, ng_fraction=0.3)
    rng = np.random.default_rng(11)
    t0 = rng.uniform(-100.0, 100.0, 70)
    t1 = t0 + rng.uniform(50.0, 250.0, 70) * np.where(np.arange(70) % 2, -1.0, 1.0)
    done, plain = _resumed(ephem, t0, t1, states, params, lanes, precision, min_dt=0.001)
    assert plain.stats.lanes_per_system == (lanes or 16) and done.stats.lanes_per_system == (lanes or 8)
    np.testing.assert_array_equal(done.steps, plain.steps)
    exact = slice(None) if precision == 0 else slice(0, 1)
    np.testing.assert_array_equal(done.states[:, exact], plain.states[:, exact])
    size = np.linalg.norm(plain.states, axis=-1)
    assert (np.linalg.norm(done.states - plain.states, axis=-1) <= 1e-12 * size).all()


@pytest.mark.parametrize("precision,metres", [(0, 0.01), (1, 1.0)])
def test_resumed_agrees_with_the_one_lane_kernel(gpu, ephem, model, precision, metres):
    """Main-belt orbits over at most 40 days (a tenth of a radian: round-off does not grow): in double
    precision a few units in the last place of 3 au a step, 1e-4 m each; the mixed form's attempts stop
    where b6 changes by 3e-9 of the acceleration, which moves a step's end by less than 1e-12 au (0.15 m)
    when round-off lets one kernel take a pass more."""
    from assist_amd import synthetic
    n = 300
    rng = np.random.default_rng(12)
    states = np.zeros((n, 1, 6))
    states[:, 0] = synthetic.main_belt(model, n, rng)
    t0 = rng.uniform(-1000.0, 1000.0, n)
    t1 = t0 + rng.uniform(20.0, 40.0, n) * np.where(np.arange(n) % 2, -1.0, 1.0)
    # (paused among the short first steps: a later boundary may be the end)
    done, plain = _resumed(ephem, t0, t1, states, None, 1, precision, at=0.02)
    assert plain.stats.lanes_per_system == 1 and done.stats.lanes_per_system == 1
    d = np.linalg.norm(done.states[:, 0, :3] - plain.states[:, 0, :3], axis=-1) * AU_M
    print("resumed against the one-lane kernel: max %.3g m" % d.max())
    assert d.max() <= metres
