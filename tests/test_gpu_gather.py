"""Rows of every length through the batched neighbour loops and tables of every
size through the staging loop, bit for bit against the oracle (FP64)."""
import numpy as np
import pytest

from jams_amd.engine import XFMT_PATTERN
from oracle import pyoracle as po
from tests import systems as S

pytestmark = pytest.mark.gpu


def chain(n, m, full, open_ends, seed=3):
    """A chain whose spin i couples to i + 1 .. i + m, one tensor per distance."""
    rng = np.random.default_rng(seed)
    J = rng.uniform(0.2, 1.0, (m, 1, 1)) * np.eye(3) if not full else rng.uniform(-1, 1, (m, 3, 3))
    pi, pj, pJ = [], [], []
    for i in range(n):
        row = sorted(((i + d) % n, d) for d in range(1, m + 1) if not open_ends or i + d < n)
        for j, d in row:
            pi.append(i)
            pj.append(j)
            pJ.append(J[d - 1].reshape(9))
    return np.array(pi, np.int32), np.array(pj, np.int32), np.array(pJ)


@pytest.mark.parametrize("full", [False, True])
@pytest.mark.parametrize("m,open_ends,block", [
    (1, False, 0), (2, False, 64), (3, True, 0), (5, False, 128), (6, True, 0), (7, False, 64),
    (9, False, 0), (12, True, 512), (15, False, 0), (40, True, 64), (100, True, 64)])
def test_row_lengths_and_table_sizes_bitwise(engine_factory, m, open_ends, block, full):
    n = 321 + 40 * m  # long enough for rows to share patterns
    pairs = chain(n, m, full, open_ends)
    csr = po.exchange_csr(n, *pairs)
    s0 = po.random_spins(5, n)
    mus, gyro, alpha = np.full(n, 2.0 * S.BOHR), np.full(n, S.gyro_e()), np.full(n, 0.1)
    o = po.OracleSystem(mus, gyro, alpha)
    o.add_exchange(*csr)
    e = engine_factory()
    e.set_sites(mus, gyro, alpha)
    e.add_exchange_csr(*csr)
    e.set_time_step(1e-3)
    e.set_exchange_format(XFMT_PATTERN)
    e.set_block_size(block)
    e.set_spins(s0)
    e.step(3)
    s = s0.copy()
    for k in range(3):
        o.heun_step(s, 1e-3, k * 1e-3)
    assert np.array_equal(e.get_spins(), s), e.describe()
