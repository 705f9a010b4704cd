"""Arrays across the C ABI: what jh_set_spins puts in, jh_get_spins gives back
bit for bit, at the sizes where the way of the copy changes (written to pinned
memory by the kernel, one chunk, several chunks on several threads) and in
both device orders."""
import numpy as np
import pytest

from oracle import pyoracle as po
from tests import systems as S

pytestmark = pytest.mark.gpu

CHUNK = 1 << 20  # bytes per staged chunk; 24 bytes per spin


@pytest.mark.parametrize("n", [1, 2, 255, 256, 257, 10922, 10923, CHUNK // 24, CHUNK // 24 + 1,
                               2 * CHUNK // 24 + 1, 16 * CHUNK // 24 - 1, 16 * CHUNK // 24 + 1,
                               17 * CHUNK // 24 + 5, 40 * CHUNK // 24 + 7])
def test_spins_round_trip(engine_factory, n):
    s = np.random.default_rng(n).standard_normal((n, 3))
    e = engine_factory()
    e.set_sites(np.ones(n), np.ones(n), np.full(n, 0.1))
    for k in range(2):
        e.set_spins(s + k)
        assert np.array_equal(e.get_spins(), s + k)
    e.close()


@pytest.mark.parametrize("L", [3, 9, 29])
def test_basis_major_order_round_trip(engine_factory, L):
    """two basis sites: the device holds the spins basis-major from L = 9"""
    b = S.c2(L, with_csr=False)
    e = engine_factory()
    e.set_sites(b.mus, b.gyro, b.alpha)
    pi, pj, pJ = b.pairs
    e.add_exchange_list(pi, pj, np.arange(pi.size, dtype=np.int32), pJ)
    e.set_time_step(b.dt)
    s = po.random_spins(3, b.n)
    e.set_spins(s)
    h = np.zeros((b.n, 3))
    np.add.at(h, pi, np.einsum("pab,pb->pa", np.asarray(pJ).reshape(-1, 3, 3), s[pj]))
    assert np.abs(e.term_field(0) - h).max() <= 1e-13 * np.abs(h).max()  # 14 terms in any order
    # (at L = 3 hardly any two rows are alike, and the order is the reference's)
    assert "order=2" in e.describe() or L == 3
    assert np.array_equal(e.get_spins(), s)
    e.set_spins(-s)
    assert np.array_equal(e.get_spins(), -s)
