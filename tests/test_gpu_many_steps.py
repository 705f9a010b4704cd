"""Small systems run many Heun steps in one launch of one workgroup: bit for
bit the two-launch kernels (which an explicit workgroup size selects), at the
smallest sizes, at wave edges and at the largest, with and without noise, in
both precision forms, across calls of any length."""
import numpy as np
import pytest

from jams_amd import configs
from jams_amd.engine import STEP_LAUNCH_PERSISTENT, XFMT_BLOCK, XFMT_TYPED
from jams_amd.host import Simulation
from oracle import pyoracle as po
from tests import systems as S

pytestmark = pytest.mark.gpu


def run(text, block, calls):
    sim = Simulation(text, device=0, output_dir="/tmp")
    e = sim.engine()
    e.set_block_size(block)
    out = []
    for n in calls:
        e.step(n)
        out.append((e.get_spins(), e.iteration(), e.magnetisation()))
    sim.close()
    return out


@pytest.mark.parametrize("precision", ["fp64", "fp32-field"])
@pytest.mark.parametrize("L,open_ends,T", [
    ((2, 1, 1), True, 5.0), ((3, 3, 7), False, 10.0), ((4, 4, 4), False, 0.0), ((5, 13, 1), True, 300.0),
    ((8, 8, 8), False, 10.0), ((8, 8, 16), False, 0.0), ((9, 9, 12), True, 20.0), ((41, 25, 1), True, 0.0)])
def test_many_steps_match_two_launches_bitwise(L, open_ends, T, precision):
    text = configs.sc_config(L=L, periodic=(not open_ends,) * 3, temperature=T, seed=9,
                             precision=precision)
    calls = (1, 2, 37, 1300)
    for (a, ia, ma), (b, ib, mb) in zip(run(text, 0, calls), run(text, 256, calls)):
        assert ia == ib
        assert np.array_equal(a, b) and np.array_equal(ma, mb)


@pytest.mark.parametrize("precision", ["fp64", "fp32-field"])
def test_two_basis_sites_and_anisotropy(precision):
    text = configs.c2(8, precision=precision)  # 1024 spins, two shells, K1, 300 K
    for (a, _, _), (b, _, _) in zip(run(text, 0, (50, 3)), run(text, 256, (50, 3))):
        assert np.array_equal(a, b)


def test_injected_noise_and_free_spins_match_the_oracle(engine_factory):
    n = 130
    b = S.c1(6)
    w = np.random.default_rng(4).standard_normal((b.n, 3))
    e = b.engine(engine_factory)
    e.set_noise(w)
    e.step(20)
    o, s = b.oracle(), b.s0.copy()
    for k in range(20):
        o.heun_step(s, b.dt, k * b.dt, w)
    assert np.array_equal(e.get_spins(), s)
    # no exchange at all
    mus, gyro, alpha = np.full(n, 2.0 * S.BOHR), np.full(n, S.gyro_e()), np.full(n, 0.1)
    dc = np.tile([0.1, 0.2, 1.0], (n, 1)) * mus[:, None]
    e = engine_factory()
    e.set_sites(mus, gyro, alpha)
    e.add_zeeman(dc)
    e.set_time_step(1e-3)
    s = po.random_spins(2, n)
    e.set_spins(s)
    e.step(30)
    o = po.OracleSystem(mus, gyro, alpha)
    o.add_zeeman(dc)
    for k in range(30):
        o.heun_step(s, 1e-3, k * 1e-3)
    assert np.array_equal(e.get_spins(), s)


@pytest.mark.parametrize("precision", ["fp64", "fp32-field"])
@pytest.mark.parametrize("L", [(3, 3, 3), (7, 7, 7), (9, 9, 9), (1023, 1, 1)])
def test_odd_numbers_of_spins(L, precision):
    """the second spin array in LDS starts behind an odd number of spins"""
    text = configs.sc_config(L=L, periodic=(False,) * 3, temperature=20.0, seed=2,
                             precision=precision)
    for (a, _, ma), (b, _, mb) in zip(run(text, 0, (1, 60)), run(text, 128, (1, 60))):
        assert np.array_equal(a, b) and np.array_equal(ma, mb)


@pytest.mark.parametrize("text,many", [
    (configs.sc_config(L=(2, 1, 1), periodic=(False,) * 3, temperature=5.0), True),
    (configs.sc_config(L=(3, 3, 7), temperature=10.0, precision="fp32-field"), True),
    (configs.sc_config(L=(5, 13, 1), periodic=(False,) * 3, temperature=300.0), True),
    (configs.sc_config(L=(8, 8, 16)), True),
    (configs.sc_config(L=(9, 9, 12), periodic=(False,) * 3, temperature=20.0), True),
    (configs.c2(8), True), (configs.c2(8, precision="fp32-field"), True),
    # one spin more than a workgroup's threads; RK4; a dipole term; power-4 anisotropy
    (configs.sc_config(L=(41, 25, 1), periodic=(False,) * 3), False),
    (configs.c1(8).replace("llg-heun-gpu", "llg-rk4-gpu"), False),
    (configs.sc_config(L=(5, 5, 3), periodic=(False,) * 3, dipole_rcut=3.0), False),
    (configs.c2(8).replace('"K1"', '"K2"'), False)])
def test_which_systems_take_the_launch(text, many):
    """the comparisons above are between two launches, and this one says which"""
    sim = Simulation(text, device=0, output_dir="/tmp")
    e = sim.engine()
    assert ("launch=many" in e.describe()) == many, e.describe()
    e.set_block_size(256)
    assert "launch=two" in e.describe()
    e.set_block_size(0)
    assert ("launch=many" in e.describe()) == many
    if many:
        e.set_step_launch(STEP_LAUNCH_PERSISTENT)
        assert "launch=persistent" in e.describe()
    sim.close()


@pytest.mark.parametrize("precision", ["fp64", "fp32-field"])
@pytest.mark.parametrize("L", [(3, 3, 3), (5, 13, 1), (7, 10, 9), (8, 8, 16)])
def test_typed_rows(L, precision):
    """tensors by id per entry instead of row patterns, and BLOCK, which keeps two launches"""
    text = configs.sc_config(L=L, periodic=(False,) * 3, temperature=20.0, seed=4,
                             precision=precision)
    got = []
    for fmt, block in ((XFMT_TYPED, 0), (XFMT_TYPED, 256), (XFMT_BLOCK, 0)):
        sim = Simulation(text, device=0, output_dir="/tmp")
        e = sim.engine()
        e.set_exchange_format(fmt)
        e.set_block_size(block)
        many = fmt == XFMT_TYPED and block == 0
        assert ("launch=many" in e.describe()) == many, e.describe()
        assert ("exchange=typed-diag" in e.describe()) == (fmt == XFMT_TYPED)
        for n in (1, 2, 70):
            e.step(n)
        got.append(e.get_spins())
        sim.close()
    assert np.array_equal(got[0], got[1])
    if precision == "fp64":
        assert np.array_equal(got[0], got[2])
