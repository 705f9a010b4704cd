"""The stage lengths of the fused dipole transforms.

The padded lengths below take every radix of the fused kernels (2 to 10, 12,
15, 16) as a single stage or as the first or last of several, on each of the
three axes, with one and several columns or lines per workgroup and with
grids from a few workgroups to several hundred.  The field is checked
against the oracle's direct offset sum with the bounds of the other dipole
tests: 1e-10 of max|h| in FP64, 1e-5 for the FP32 transforms.
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
