"""The stage lengths of the dipole transforms.

Between them the lengths below take every radix of the fused kernels (2 to 10,
12, 15, 16) along x and along y, alone and as the first or last of several,
and lengths of 1, which have no stages; z is a direct transform in the fused
kernels.  The first set of lattices also has two basis sites, long z axes and
lengths that the separate passes take, with one and several columns or lines
per workgroup and grids from a few workgroups to several hundred.  The field
is checked against the oracle's direct offset sum with the bounds of the other
dipole tests: 1e-10 of max|h| in FP64, 1e-5 for the FP32 transforms.
"""
import numpy as np
import pytest

from oracle import pyoracle as po
from tests.test_gpu_dipole import A, SC, dipole_engine, rnd_spins
from tests import systems as S

pytestmark = pytest.mark.gpu

ONE = [[0, 0, 0]]
TWO = [[0, 0, 0], [0.5, 0.5, 0.5]]

CASES = [
    ("p6_p9_p10", (6, 9, 10), (1, 1, 1), ONE, 2.9),
    ("p7_p12_p15", (7, 12, 15), (1, 1, 1), ONE, 3.4),
    ("p16_p14_p21", (16, 14, 21), (1, 1, 1), ONE, 5.0),
    ("p15_p35_p16", (15, 35, 16), (1, 1, 1), ONE, 5.0),
    ("p21_p16_p7_two_sites", (21, 16, 7), (1, 1, 1), TWO, 3.2),
    ("p49_p10_open9", (49, 10, 9), (1, 1, 0), ONE, 4.5),
    ("open49_open63_open3", (49, 63, 3), (0, 0, 0), ONE, 12.0),
    ("open90_open75_open3", (90, 75, 3), (0, 0, 0), ONE, 6.0),
    ("open1_open72_open56", (1, 72, 56), (0, 0, 0), ONE, 30.0),
    ("p240_p60_open2", (240, 60, 2), (1, 1, 0), ONE, 4.0),
]


@pytest.mark.parametrize("name,size,per,basis,rc", CASES, ids=[c[0] for c in CASES])
def test_dipole_field_of_each_radix(engine_factory, name, size, per, basis, rc):
    lat = po.LatticeSpec(SC, basis, list(range(len(basis))), size, per)
    mus = np.where(np.arange(lat.n) % len(basis) == 0, 2.3, 1.7) * S.BOHR
    s = rnd_spins(lat.n, 23)
    ref = po.dipole_fft_direct(lat, mus, s, rc, A, nthreads=8)
    scale = np.abs(ref).max()
    err = {}
    for prec in (0, 1):
        e = dipole_engine(engine_factory, lat, mus, rc, prec=prec)
        e.set_spins(s)
        err[prec] = np.abs(e.term_field(0) - ref).max() / scale
    print(f"{name}: max|h| {scale:.3e} meV, rel err FP64 {err[0]:.2e}, FP32 {err[1]:.2e}")
    assert err[0] <= 1e-10
    assert err[1] <= 1e-5


FUSED = [(8, 9, 2), (9, 8, 2), (10, 4, 2), (4, 10, 2), (5, 3, 2), (3, 5, 2), (6, 7, 2), (7, 6, 2),
         (12, 15, 3), (15, 12, 3), (16, 2, 2), (2, 16, 2), (72, 20, 2), (20, 72, 2), (64, 27, 1),
         (27, 64, 1), (80, 45, 5), (45, 80, 5), (14, 32, 4), (32, 14, 4), (128, 96, 1),
         (96, 128, 1), (1, 9, 4), (8, 1, 4), (1, 1, 20), (9, 1, 1), (1, 12, 1), (300, 1, 8),
         (1, 512, 2), (512, 1, 2)]


@pytest.mark.parametrize("size", FUSED, ids=lambda s: "x".join(map(str, s)))
def test_fused_kernels_at_every_radix(engine_factory, size):
    """one basis site, x and y periodic (no padding), z open"""
    lat = po.LatticeSpec(SC, ONE, [0], size, (1, 1, 0))
    mus = np.full(lat.n, 2.3 * S.BOHR)
    s = rnd_spins(lat.n, 31)
    rc = max(1.3, min(6.0, 0.45 * min(size[:2])))
    ref = po.dipole_fft_direct(lat, mus, s, rc, A, nthreads=8)
    scale = np.abs(ref).max()
    for prec, bound in ((0, 1e-10), (1, 1e-5)):
        e = dipole_engine(engine_factory, lat, mus, rc, prec=prec)
        e.set_spins(s)
        d = e.describe()
        assert "dip_x=fused" in d and "dip_zyf=fused" in d and "dip_zyi=fused" in d, d
        assert np.abs(e.term_field(0) - ref).max() <= bound * scale
