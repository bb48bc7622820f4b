"""The kernel that a launch without overrides takes follows from the batch alone, whatever ran before it in
the process: real-only batches of 131,072 systems or more run on one lane per system, unless their spans are
so uneven that the launch would end on a few costly ones.  Main-belt
orbits over at most 20 days, on which the kernels differ by round-off alone: steps of days, each leaving a
few units in the last place of 3 au (1e-4 m each), so 1 cm holds many of them, and a wrong record, body or
hand-over moves a position by kilometres."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
AU_M = 149597870700.0
N = 131072 + 65


@pytest.fixture(scope="module")
def belt(model):
    from assist_amd import synthetic
    states = np.zeros((N, 1, 6))
    states[:, 0] = synthetic.main_belt(model, N, np.random.default_rng(61))
    return states


@pytest.mark.parametrize("forces", [0x7F, 0x5F])
@pytest.mark.parametrize("precision", [0, 1])
def test_default_choice_does_not_depend_on_earlier_calls(gpu, ephem, belt, precision, forces):
    """A first call whose spans are all zero, then one of 20 days: one lane per system, with the bits of
    lanes_per_system = 1, and within round-off of the 8-lane kernel."""
    from assist_amd import batch
    ex = {"forces": forces}
    cfg = batch.BatchConfig.default(precision=precision)
    t1 = np.random.default_rng(62).uniform(-20.0, 20.0, N)
    zero = batch.integrate(ephem, 0.0, np.zeros(N), belt, extras=ex, config=cfg)
    assert zero.stats.lanes_per_system == 1 and zero.stats.block_size == 256
    np.testing.assert_array_equal(zero.states, belt)
    auto = batch.integrate(ephem, 0.0, t1, belt, extras=ex, config=cfg)
    one = batch.integrate(ephem, 0.0, t1, belt, extras=ex,
                          config=batch.BatchConfig.default(precision=precision, lanes_per_system=1))
    assert auto.stats.lanes_per_system == 1 and auto.stats.block_size == 256 and (auto.status == 0).all()
    for k in ("states", "status", "steps"):
        np.testing.assert_array_equal(getattr(auto, k), getattr(one, k))
    groups = batch.integrate(ephem, 0.0, t1, belt, extras=ex,
                             config=batch.BatchConfig.default(precision=precision, lanes_per_system=8))
    assert (groups.status == 0).all()
    d = np.linalg.norm(auto.states[:, 0, :3] - groups.states[:, 0, :3], axis=-1) * AU_M
    assert d.max() <= (0.01 if precision == 0 else 1.0)


@pytest.mark.parametrize("precision", [0, 1])
def test_uneven_spans_take_16_lanes(gpu, ephem, belt, precision):
    """One span in a hundred is 100 days, the others half a day: all steps together are 50,000 times the
    costliest system's (one lane); with 3,000 days, 3,400 times.  On 16 lanes the bits are the 8-lane
    kernel's."""
    from assist_amd import batch
    for long, lanes in ((100.0, 1), (3000.0, 16)):
        t1 = np.full(N, 0.5)
        t1[::100] = -long
        r = batch.integrate(ephem, 0.0, t1, belt, config=batch.BatchConfig.default(precision=precision))
        assert r.stats.lanes_per_system == lanes and (r.status == 0).all()
        if lanes == 16:
            groups = batch.integrate(ephem, 0.0, t1, belt,
                                     config=batch.BatchConfig.default(precision=precision, lanes_per_system=8))
            np.testing.assert_array_equal(r.states, groups.states)
            np.testing.assert_array_equal(r.steps, groups.steps)


def test_below_the_line_16_lanes(gpu, ephem, belt):
    from assist_amd import batch
    r = batch.integrate(ephem, 0.0, 1.0, belt[:131071])
    assert r.stats.lanes_per_system == 16 and (r.status == 0).all()
