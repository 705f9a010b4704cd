"""Small contexts replay a graph of their own accord after enough
plain steps: the same bits as calls too short for a replay, replay after
replay, with reductions, field evaluations and set-up changes in between."""
import ctypes
import subprocess
import sys
import threading
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

import numpy as np
import pytest

from jams_amd import configs
from jams_amd.host import Simulation

pytestmark = pytest.mark.gpu

F32 = "fp32-field"
CASES = {
    "heun": configs.sc_config(L=(13, 11, 12), temperature=20.0, seed=3),
    "heun fp32": configs.sc_config(L=(13, 11, 12), temperature=20.0, seed=3, precision=F32),
    "rk4": configs.bcc_config(L=9, seed=5).replace("llg-heun-gpu", "llg-rk4-gpu"),
    "two shells": configs.bcc_config(L=9, seed=5),
    "film": configs.sc_config(L=(14, 10, 3), periodic=(False,) * 3, field=None, dipole_rcut=20.0,
                              alpha=0.02),
    "film fp32": configs.sc_config(L=(14, 10, 3), periodic=(False,) * 3, field=None,
                                   dipole_rcut=20.0, alpha=0.02, precision=F32),
}


def steps(e, n, most):
    while n > 0:
        e.step(min(n, most))
        n -= most


@pytest.mark.parametrize("name", CASES)
def test_replays_match_short_calls_bitwise(name):
    sims = [Simulation(CASES[name], device=0, output_dir="/tmp") for _ in range(2)]
    a, b = (s.engine() for s in sims)
    for k, n in enumerate((510, 100, 7, 45, 200)):
        steps(a, n, 19)      # shorter than a replay: plain launches
        steps(b, n, 10_000)
        assert a.iteration() == b.iteration()
        assert np.array_equal(a.get_spins(), b.get_spins()), (name, k)
        assert np.array_equal(a.magnetisation(), b.magnetisation())
        b.fields()
        b.magnetisation()
    # injected noise replaces the stream that the graph holds
    w = np.random.default_rng(1).standard_normal((a.n, 3))
    for e, most in ((a, 19), (b, 10_000)):
        e.set_noise(w)
        steps(e, 60, most)
    assert np.array_equal(a.get_spins(), b.get_spins())
    # and so does a new time step
    for e, most in ((a, 19), (b, 10_000)):
        e.set_time_step(5e-4)
        steps(e, 560, most)
    assert np.array_equal(a.get_spins(), b.get_spins())
    for s in sims:
        s.close()


def test_describe_tells_the_graph():
    sim = Simulation(CASES["heun"], device=0, output_dir="/tmp")
    e = sim.engine()
    assert "graph=0 " in e.describe()
    e.step(499)
    assert "graph=0 " in e.describe()
    e.step(1)
    assert "graph=20 " in e.describe()
    e.set_graph_steps(7)
    assert "graph=7 " in e.describe()
    e.set_graph_steps(0)
    e.step(600)
    assert "graph=0 " in e.describe()
    sim.close()


@pytest.mark.parametrize("chosen", [0, 20])
def test_noise_set_before_every_few_steps(chosen):
    """New values in the same buffer keep the graph, the engine's own and the
    caller's; only the first ones, or another workgroup size, end it."""
    a, b = (Simulation(CASES["heun"], device=0, output_dir="/tmp") for _ in range(2))
    e, f = a.engine(), b.engine()
    if chosen:
        e.set_graph_steps(chosen)
    e.step(600)
    f.set_graph_steps(0)
    f.step(600)
    rng = np.random.default_rng(8)
    for k in range(40):
        w = rng.standard_normal((e.n, 3))
        for q in (e, f):
            q.set_noise(w)
            q.step(20)
        assert (f"graph={20 if chosen or k > 24 else 0} " in e.describe()) or k == 24, k
    assert np.array_equal(e.get_spins(), f.get_spins())
    e.set_block_size(128)
    assert f"graph={chosen} " in e.describe()
    for q in (e, f):
        q.step(100)
    assert np.array_equal(e.get_spins(), f.get_spins())
    a.close()
    b.close()


def test_contexts_on_several_threads():
    """Each thread sets contexts up, steps them past the point where they build
    a graph and reads them, while the others do the same: the bits of the same
    runs one after the other."""
    texts = [configs.sc_config(L=(13, 11, 12), temperature=20.0, seed=3),
             configs.sc_config(L=(13, 11, 12), temperature=20.0, seed=4, precision=F32),
             configs.bcc_config(L=9, seed=5), CASES["film"]]

    def go(text):
        out = []
        for _ in range(6):
            s = Simulation(text, device=0, output_dir="/tmp")
            e = s.engine()
            for n in (490, 30, 75):
                e.step(n)
                out.append(e.get_spins())
            e.set_thermostat(5.0, 9)
            e.step(560)
            out.append(e.get_spins())
            out.append(e.magnetisation())
            s.close()
        return out

    alone = [go(t) for t in texts]
    with ThreadPoolExecutor(len(texts)) as pool:
        together = list(pool.map(go, texts))
    for a, b in zip(alone, together):
        assert len(a) == len(b) and all(np.array_equal(x, y) for x, y in zip(a, b))


def test_building_a_graph_leaves_other_threads_alone():
    """Copies on the legacy stream by another thread of the process, which a
    stream capture anywhere in it would have the runtime refuse."""
    sim = Simulation(CASES["heun"], device=0, output_dir="/tmp")
    e = sim.engine()
    hip = e.lib  # the engine's own HIP library is found through it
    dev, host = ctypes.c_void_p(), (ctypes.c_char * 64)()
    assert hip.hipMalloc(ctypes.byref(dev), ctypes.c_size_t(64)) == 0
    done, results = threading.Event(), []

    def copy():
        while not done.is_set():
            results.append(hip.hipMemcpy(dev, host, ctypes.c_size_t(64), 1))

    t = threading.Thread(target=copy)
    t.start()
    try:
        for k in range(20):
            e.set_graph_steps(300 + k)
            e.step(300 + k)
    finally:
        done.set()
        t.join()
    e.synchronize()
    assert hip.hipFree(dev) == 0
    assert len(results) > 20 and not any(results)
    sim.close()


CHILD = """
import ctypes, sys
ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)  # before the engine's own HIP library
import numpy as np
from jams_amd import configs
from jams_amd.engine import EngineError
from jams_amd.host import Simulation
a, b = (Simulation(configs.c1(16, temperature=10.0), device=0, output_dir="/tmp") for _ in range(2))
for s, most in ((a, 19), (b, 700)):
    e, n = s.engine(), 1400
    while n > 0:
        e.step(min(n, most))
        n -= most
assert np.array_equal(a.engine().get_spins(), b.engine().get_spins())
e = a.engine()
print(b.engine().autotune(40))
e.set_graph_steps(20)
try:
    e.step(20)
except EngineError as err:
    print("CHILD OK", err)
"""


def test_steps_run_plainly_where_no_graph_is_to_be_had(tmp_path):
    """hipGraphInstantiate replaced by one that always fails: a graph that the
    engine chose by itself is given up, one that the caller asked for is an error"""
    src = tmp_path / "nograph.c"
    src.write_text("int hipGraphInstantiate(void *e, void *g, void *n, char *b, unsigned long s)"
                   "{ *(void **)e = 0; return 2; }\n")
    lib = tmp_path / "nograph.so"
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", str(lib), str(src)], check=True)
    r = subprocess.run([sys.executable, "-c", CHILD, str(lib)], capture_output=True, text=True,
                       cwd=Path(__file__).resolve().parents[1], timeout=100)
    assert r.returncode == 0 and "CHILD OK" in r.stdout, r.stdout + r.stderr
