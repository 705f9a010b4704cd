"""jh_step returns before its launches have run.  A change of the set-up, of the
launch shape or of the graph length right behind it waits for them: the same
bits as with a jh_synchronize in between."""
import numpy as np
import pytest

from oracle import pyoracle as po
from tests import systems as S

pytestmark = pytest.mark.gpu


def alloy(engine_factory, L):
    """open simple cubic, two materials: several site classes, tables that hold
    the thermostat's and the time step's factors"""
    n = L ** 3
    kind = (np.random.default_rng(2).random(n) < 0.4).astype(np.int32)
    index = np.arange(n, dtype=np.int32).reshape(L, L, L)
    pi, pj = [], []
    for ax in range(3):
        a = np.take(index, np.arange(L - 1), ax).reshape(-1)
        b = np.take(index, np.arange(1, L), ax).reshape(-1)
        pi += [a, b]
        pj += [b, a]
    i, j = np.concatenate(pi), np.concatenate(pj)
    order = np.lexsort((j, i))
    i, j = i[order], j[order]
    e = engine_factory()
    e.set_sites(np.where(kind == 0, 2.2, 1.6) * S.BOHR, np.full(n, S.gyro_e()),
                np.where(kind == 0, 0.02, 0.05))
    e.add_exchange_list(i, j, 2 * kind[i] + kind[j],
                        np.stack([v * np.eye(3) for v in (2.0, -1.0, -1.0, 1.2)]))
    e.set_time_step(1e-3)
    e.set_thermostat(10.0, 3)
    e.set_spins(po.random_spins(4, n))
    return e


@pytest.mark.parametrize("L", [6, 30])
def test_changes_behind_queued_steps(engine_factory, L):
    changes = [lambda e: e.set_thermostat(300.0, 5), lambda e: e.set_time_step(5e-4),
               lambda e: e.set_block_size(128), lambda e: e.set_block_size(0),
               lambda e: e.set_graph_steps(40), lambda e: e.set_graph_steps(0),
               lambda e: e.set_noise(po.random_spins(6, e.n))]
    a, b = alloy(engine_factory, L), alloy(engine_factory, L)
    for k, change in enumerate(changes):
        for e, wait in ((a, True), (b, False)):
            e.step(900)
            if wait:
                e.synchronize()
            change(e)
            e.step(25)
        assert np.array_equal(a.get_spins(), b.get_spins()), k
