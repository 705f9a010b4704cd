"""The thermostat's normal deviates at the corners of its counter (large steps
and seeds, few and many spins) bit for bit against the oracle's stream."""
import numpy as np
import pytest

from oracle import pyoracle as po
from tests import systems as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("seed,step,n", [
    (0, 0, 1), (2**64 - 1, 2**32 - 1, 65), (0x8000000180000001, 2**32, 4097),
    (1, (1 << 52) + 3, 300_001)])
def test_noise_stream_corners_bitwise(engine_factory, seed, step, n):
    mus, gyro, alpha = np.full(n, 2.0 * S.BOHR), np.full(n, S.gyro_e()), np.full(n, 0.1)
    e = engine_factory()
    e.set_sites(mus, gyro, alpha)
    e.set_spins(np.tile([0.0, 0.0, 1.0], (n, 1)))
    e.set_time_step(1e-3)
    e.set_thermostat(300.0, seed)
    ref = po.scale_noise(po.normals(seed, step, n), po.thermostat_sigma(mus, gyro, alpha, 1e-3), 300.0)
    assert np.array_equal(e.get_noise(step), ref)
