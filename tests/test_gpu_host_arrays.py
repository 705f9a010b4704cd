"""Arrays across the C ABI: what jh_set_spins puts in, jh_get_spins gives back
bit for bit, at the sizes where the way of the copy changes (written to pinned
memory by the kernel, one chunk, several chunks on several threads) and in
both device orders."""
import ctypes
import subprocess
import sys
from pathlib import Path

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


def test_no_device_memory_for_the_transfers(engine_factory):
    """s, s*, ds and the field output: four arrays of 24 bytes per spin, and the
    transfers take no fifth one"""
    def free_bytes():
        free, total = ctypes.c_size_t(), ctypes.c_size_t()
        assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
        return free.value

    n = 1 << 22
    e = engine_factory()
    hip = e.lib  # the engine's own HIP library is found through it
    before = free_bytes()
    e.set_sites(np.ones(n), np.ones(n), np.full(n, 0.1))
    s = np.random.default_rng(3).standard_normal((n, 3))
    e.set_spins(s)
    assert np.array_equal(e.get_spins(), s)
    assert before - free_bytes() <= 4 * 24 * n + (16 << 20)


def test_reads_between_steps_leave_them_alone(engine_factory):
    """spins, fields and noise read back between steps of both integrators, and
    the steps that follow, against a context that is not read"""
    for integrator in (0, 1):
        b = S.c2(24)
        got = []
        for reads in (True, False):
            e = b.engine(engine_factory)
            e.set_integrator(integrator)
            e.set_thermostat(300.0, 7)
            for _ in range(3):
                e.step(2)
                if reads:
                    s = e.get_spins()
                    h = e.fields()
                    w = e.get_noise(1)
                    assert np.array_equal(h, e.fields()) and np.array_equal(w, e.get_noise(1))
                    assert np.array_equal(s, e.get_spins())
            got.append(e.get_spins())
        assert np.array_equal(*got)


CHILD = """
import ctypes, sys, threading
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)  # before the engine's own HIP library
import numpy as np
from jams_amd import configs
from jams_amd.host import Simulation
sim = Simulation(configs.sc_config(L=(40, 40, 40), temperature=10.0), device=0, output_dir="/tmp")
e = sim.engine()
e.step(1)
s = e.get_spins()
for call in (e.get_spins, lambda: e.set_spins(s), e.fields, lambda: e.get_noise(1),
             lambda: e.set_noise(s)):
    before = shim.calls()
    t = threading.Thread(target=call)
    t.start()
    t.join()
    assert shim.calls() > before
print("CHILD OK")
"""


def test_transfers_bind_the_context_s_device(tmp_path):
    """A thread whose current device is another one reads and sets arrays: each
    transfer selects the context's device (counted by a hipSetDevice that
    stands in for the library's; the one device is current anyway)."""
    src = tmp_path / "device.c"
    src.write_text("static int n; int hipSetDevice(int d) { __sync_fetch_and_add(&n, 1); return d != 0; }"
                   " int calls(void) { return n; }\n")
    lib = tmp_path / "device.so"
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", str(lib), str(src)], check=True)
    r = subprocess.run([sys.executable, "-c", CHILD, str(lib)], capture_output=True, text=True,
                       cwd=Path(__file__).resolve().parents[1], timeout=100)
    assert r.returncode == 0 and "CHILD OK" in r.stdout, r.stdout + r.stderr
