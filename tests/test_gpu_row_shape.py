"""Launch shape of the 16-lane kernel: above four systems per SIMD, blocks of three waves where its
registers hold two waves per SIMD, and of four where they hold one, so that no SIMD of a CU stays
without work; the stats tell which it is."""
import numpy as np
import pytest

from conftest import population

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_var,marsden,forces,precision,waves", [
    (7, True, 0x7F, 0, 1), (3, True, 0x7F, 0, 1), (6, False, 0x3F, 0, 1), (2, False, 0x3F, 0, 1),
    (6, False, 0x7F, 0, 2), (3, True, 0x7F, 1, 2), (7, True, 0x3F, 1, 2), (0, True, 0x7F, 0, 2), (0, False, 0x3F, 0, 2)])
def test_blocks_fill_the_simds(gpu, ephem, model, n_var, marsden, forces, precision, waves):
    from assist_amd import batch
    n = 6151
    states, params, _ = population(model, n, 71 + n_var, n_var=n_var, ng_fraction=0.3)
    params = params if marsden else None
    t1 = np.where(np.arange(n) % 2, -3.0, 5.0)
    got = batch.integrate(ephem, 0.0, t1, states, params, extras={"forces": forces},
                          config=batch.BatchConfig.default(precision=precision, min_dt=0.001))
    ref = batch.integrate(ephem, 0.0, t1, states, params, extras={"forces": forces},
                          config=batch.BatchConfig.default(precision=precision, min_dt=0.001, lanes_per_system=8))
    assert got.stats.lanes_per_system == 16 and got.stats.waves_per_simd == waves
    assert got.stats.block_size == (256 if waves == 1 else 192)
    np.testing.assert_array_equal(got.states, ref.states)
    np.testing.assert_array_equal(got.steps, ref.steps)


@pytest.mark.parametrize("n,threads", [(1, 64), (1024, 64), (1025, 256), (4096, 256), (4097, 192)])
def test_blocks_by_size(gpu, ephem, model, n, threads):
    """The lines on a chip of 256 CUs."""
    from assist_amd import batch
    states, _, _ = population(model, n, 81, n_var=6)
    r = batch.integrate(ephem, 0.0, 0.5, states)
    assert (r.status == 0).all() and r.stats.block_size == threads and r.stats.waves_per_simd == 2
