"""The work a user of this framework has it do, as cases that can be timed.

Every case is one stretch of a spin-dynamics run as a JAMS program makes it:
the context (lattice, exchange, thermostat) is set up once and kept, and a
pass advances it by `steps` time steps and then reads what monitors read, the
spins and the summed moments.  100 steps between readings is the default
`output_steps` of the monitors.

    listed()           the cases
    draw(rng)          one more of the ranges they stand for
    prepare(case, seed), run(state), work(case)
    exact(case, seed)  the same outputs in 64-bit torch, from the equations
"""
from __future__ import annotations

import math
import tempfile

import numpy as np
import torch

from jams_amd import configs
from jams_amd.batch import ReplicaBatch
from jams_amd.engine import INTEGRATOR_RK4, PREC_FP32_FIELD, Engine
from jams_amd.host import Simulation

# internal units: energies meV, fields T, times ps (helpers/consts.h:18-38)
BOHR = 0.0578838181
GYRO = 2.0023193043625 * 0.0578838181 / 0.6582119569
KB = 0.0861733326
MU0 = 4.0 * math.pi * 1e-7 / 6.24150907e21
ALLOY_J = {(0, 0): 2.0, (0, 1): -1.0, (1, 0): -1.0, (1, 1): 1.2}


def listed():
    return [
        # the smallest runs (unit tests of a material, parameter fits): a step
        # is a few microseconds and launches are what counts
        {"name": "sc 8^3", "kind": "sc", "x": 8, "y": 8, "z": 8, "open": False, "T": 0.0,
         "precision": "fp64", "integrator": "heun", "steps": 100},
        # the 16^3 validation system, with its thermostat on
        {"name": "sc 16^3 langevin", "kind": "sc", "x": 16, "y": 16, "z": 16, "open": False,
         "T": 10.0, "precision": "fp64", "integrator": "heun", "steps": 100},
        # an ordinary production size: bcc 64^3 x 2, two shells, 300 K, in both
        # precision forms and with the other integrator
        {"name": "bcc 64^3 two shells", "kind": "bcc2", "x": 64, "y": 64, "z": 64, "open": False,
         "T": 300.0, "precision": "fp64", "integrator": "heun", "steps": 100},
        {"name": "bcc 64^3 two shells fp32-field", "kind": "bcc2", "x": 64, "y": 64, "z": 64,
         "open": False, "T": 300.0, "precision": "fp32-field", "integrator": "heun",
         "steps": 100},
        {"name": "bcc 64^3 two shells rk4", "kind": "bcc2", "x": 64, "y": 64, "z": 64,
         "open": False, "T": 300.0, "precision": "fp64", "integrator": "rk4", "steps": 100},
        # the headline: 4.2 million spins, 58 neighbours with DMI (full tensors)
        {"name": "bcc 128^3 five shells", "kind": "bcc5", "x": 128, "y": 128, "z": 128,
         "open": False, "T": 100.0, "precision": "fp64", "integrator": "heun", "steps": 100},
        # the same material at ordinary sizes: in the FP32-field form, and a
        # supercell whose sides are no powers of two
        {"name": "bcc 64^3 five shells fp32-field", "kind": "bcc5", "x": 64, "y": 64, "z": 64,
         "open": False, "T": 100.0, "precision": "fp32-field", "integrator": "heun",
         "steps": 100},
        {"name": "bcc 36x33x35 five shells", "kind": "bcc5", "x": 36, "y": 33, "z": 35,
         "open": False, "T": 100.0, "precision": "fp64", "integrator": "heun", "steps": 100},
        # a temperature and field sweep as one batch of independent systems
        # (8^3 to 48^3 spins each), stepped by graph replays
        {"name": "64 replicas", "kind": "replicas", "n": 64, "precision": "fp64", "steps": 100},
        # thin films with the dipole field: the large square one, and a small
        # ragged one with FP32 transforms
        {"name": "film 256x256x8", "kind": "film", "x": 256, "y": 256, "z": 8,
         "precision": "fp64", "steps": 100},
        {"name": "film 90x75x6 fp32-field", "kind": "film", "x": 90, "y": 75, "z": 6,
         "precision": "fp32-field", "steps": 100},
        # a random alloy (two materials) with open boundaries and odd sides:
        # no two rows alike, tensors by table
        {"name": "alloy 61x53x47", "kind": "alloy", "x": 61, "y": 53, "z": 47, "T": 40.0,
         "precision": "fp64", "steps": 100},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _fft_side(rng, lo, hi):
    """a film side as one picks it for a Fourier grid (prime factors 2, 3, 5 and 7)"""
    while True:
        n = m = _log_int(rng, lo, hi)
        for f in (2, 3, 5, 7):
            while m % f == 0:
                m //= f
        if m == 1:
            return n


def draw(rng):
    kind = rng.choice(["sc", "sc", "bcc2", "bcc2", "bcc5", "bcc5", "replicas", "film", "film",
                       "alloy"])
    precision = rng.choice(["fp64", "fp64", "fp32-field"])
    if kind == "sc":
        x, y, z = (_log_int(rng, 6, 72) for _ in range(3))
        return {"kind": kind, "x": x, "y": y, "z": z, "open": rng.random() < 0.3,
                "T": rng.choice([0.0, 10.0, 300.0]), "precision": precision,
                "integrator": rng.choice(["heun", "heun", "heun", "rk4"]), "steps": 100}
    if kind == "bcc2":
        x, y, z = (_log_int(rng, 10, 80) for _ in range(3))
        return {"kind": kind, "x": x, "y": y, "z": z, "open": rng.random() < 0.2,
                "T": rng.choice([0.0, 300.0]), "precision": precision,
                "integrator": rng.choice(["heun", "heun", "heun", "rk4"]), "steps": 100}
    if kind == "bcc5":
        x, y = (_log_int(rng, 12, 64) for _ in range(2))
        z = 64 if rng.random() < 0.5 else _log_int(rng, 12, 70)
        return {"kind": kind, "x": x, "y": y, "z": z, "open": rng.random() < 0.15, "T": 100.0,
                "precision": precision, "integrator": "heun", "steps": 100}
    if kind == "replicas":
        return {"kind": kind, "n": _log_int(rng, 8, 80), "precision": precision, "steps": 100}
    if kind == "film":
        return {"kind": kind, "x": _fft_side(rng, 24, 256), "y": _fft_side(rng, 24, 256),
                "z": rng.randint(1, 8), "precision": precision, "steps": 100}
    x, y, z = (_log_int(rng, 9, 72) for _ in range(3))
    return {"kind": kind, "x": x, "y": y, "z": z, "T": 40.0, "precision": precision,
            "steps": 100}


# ---------------------------------------------------------------------------
# the systems

def _material(case):
    """exchange rows, basis, moment (muB), alpha, dt (s), field (T), K1 (meV)"""
    k = case["kind"]
    if k == "sc":
        return configs.sc_neighbour_rows(1.0), 1, 2.0, 0.1, 1e-15, (0.0, 0.0, 1.0), None
    if k == "film":
        return configs.sc_neighbour_rows(2.0), 1, 2.2, 0.02, 1e-15, None, None
    if k == "bcc2":
        return configs.bcc_two_shell_rows(3.0, 1.5), 2, 2.0, 0.05, 0.5e-15, None, 0.05
    return configs.bcc_five_shell_dmi_rows(), 2, 2.0, 0.05, 0.5e-15, None, None


def _film_cutoff(case):
    # the longest diagonal: every pair of the film interacts
    return math.sqrt(case["x"] ** 2 + case["y"] ** 2 + case["z"] ** 2)


def _text(case, seed):
    """The JAMS config of an sc, bcc or film case."""
    rows, nb, moment, alpha, dt, field, K = _material(case)
    per = "false" if case["kind"] == "film" or case.get("open") else "true"
    positions = '("A", [0.0, 0.0, 0.0])' + (', ("A", [0.5, 0.5, 0.5])' if nb == 2 else "")
    ham = ['{ module = "exchange"; energy_units = "meV"; symops = false; '
           f"interactions = ( {configs.interactions_text(rows)} ); }}"]
    if field is not None:
        ham.append(f'{{ module = "applied-field"; field = [{field[0]}, {field[1]}, {field[2]}]; }}')
    if K is not None:
        ham.append('{ module = "uniaxial"; order = "K1"; energy_units = "meV"; '
                   f'anisotropies = ( ("A", [0.0, 0.0, 1.0], {K!r}) ); }}')
    if case["kind"] == "film":
        ham.append(f'{{ module = "dipole-fft"; r_cutoff = {_film_cutoff(case)!r}; }}')
    module = "llg-rk4-gpu" if case.get("integrator") == "rk4" else "llg-heun-gpu"
    return f"""
materials = ( {{ name = "A"; moment = {moment!r}; alpha = {alpha!r}; gyro = 1.0; spin = [0.0, 0.0, 1.0]; }} );
unitcell : {{ parameter = 0.3e-9; symops = false; positions = ( {positions} );
  basis = ([1.0, 0.0, 0.0], [0.0, 1.0, 0.0], [0.0, 0.0, 1.0]); }};
lattice : {{ size = [{case["x"]}, {case["y"]}, {case["z"]}]; periodic = [{per}, {per}, {per}]; }};
hamiltonians = ( {", ".join(ham)} );
solver : {{ module = "{module}"; t_step = {dt!r}; t_max = {dt * 1000!r}; precision = "{case["precision"]}"; }};
physics : {{ temperature = {float(case.get("T", 0.0))!r}; }};
sim : {{ seed = {seed}; }};
"""


def _spins(n, seed):
    """n unit vectors, uniform on the sphere, from the seed alone"""
    s = np.random.default_rng(seed).standard_normal((n, 3))
    s /= np.sqrt((s * s).sum(1))[:, None]
    return s


def _alloy(case, seed):
    """Site types and, per direction, (site, neighbour) pairs of an open sc alloy."""
    size = (case["x"], case["y"], case["z"])
    types = (np.random.default_rng(seed + 7).random(size) < 0.3).astype(np.int32).reshape(-1)
    index = np.arange(types.size, dtype=np.int32).reshape(size)
    pi, pj = [], []
    for ax in range(3):
        a = np.take(index, np.arange(size[ax] - 1), ax).reshape(-1)
        b = np.take(index, np.arange(1, size[ax]), ax).reshape(-1)
        pi += [a, b]
        pj += [b, a]
    return types, pi, pj


def _alloy_sites(types):
    mus = np.where(types == 0, 2.2, 1.6) * BOHR
    alpha = np.where(types == 0, 0.02, 0.05)
    return mus, np.full(types.size, GYRO), alpha


def _replicas(case, seed):
    """(text, T, noise seed, field, description) per replica; the sizes are the
    sweep's own and do not change with the seed"""
    reps = configs.c4(case["n"], precision=case["precision"], steps=1000)
    return [(text, T, seed * 1000 + r, B, desc) for r, (text, T, _, B, desc) in enumerate(reps)]


def prepare(case, seed):
    prec = PREC_FP32_FIELD if case["precision"] == "fp32-field" else 0
    state = {"steps": case["steps"], "kind": case["kind"]}
    if case["kind"] == "replicas":
        batch = ReplicaBatch(_replicas(case, seed), precision=prec, output_dir=tempfile.gettempdir())
        e = batch.engine
        e.set_graph_steps(50)
        state["keep"] = batch
    elif case["kind"] == "alloy":
        types, pi, pj = _alloy(case, seed)
        i, j = np.concatenate(pi), np.concatenate(pj)
        order = np.lexsort((j, i))
        i, j = i[order], j[order]
        e = Engine(0)
        e.set_sites(*_alloy_sites(types))
        values = np.stack([ALLOY_J[p] * np.eye(3) for p in ((0, 0), (0, 1), (1, 0), (1, 1))])
        e.add_exchange_list(i, j, 2 * types[i] + types[j], values)
        e.set_time_step(1e-3)
        e.set_precision(prec)
        e.set_thermostat(case["T"], seed)
    else:
        sim = Simulation(_text(case, seed), device=0, output_dir=tempfile.gettempdir())
        e = sim.engine()
        state["keep"] = sim
    e.set_spins(_spins(e.n, seed))
    # monitors are notified before the first step
    _moments(state, e)
    state["engine"] = e
    return state


def _moments(state, e):
    if state["kind"] == "replicas":
        return state["keep"].engine.replica_magnetisation()
    return e.magnetisation()


def run(state):
    e = state["engine"]
    e.step(state["steps"])
    out = {"spins": e.get_spins(), "moments": _moments(state, e)}
    if state["kind"] == "alloy":
        out["energy"] = np.array([e.term_energy(0)])
    return out


# ---------------------------------------------------------------------------
# what a pass cannot do without

def work(case):
    k = case["kind"]
    if k == "replicas":
        n = sum(_replica_size(case)[1])
        nbrs, diag = 7.0, True
    else:
        n = case["x"] * case["y"] * case["z"] * (2 if k in ("bcc2", "bcc5") else 1)
        nbrs = {"sc": 6.0, "film": 6.0, "alloy": 6.0, "bcc2": 14.0, "bcc5": 58.0}[k]
        diag = k != "bcc5"
    evals = 4 if case.get("integrator") == "rk4" else 2
    # per evaluation: the exchange sum, h / mus, the LLG right-hand side and
    # the update with its renormalisation; per thermal step three normals
    flops = evals * (nbrs * (6.0 if diag else 18.0) + 60.0)
    if k == "replicas" or case.get("T", 0.0) > 0.0:
        flops += 130.0
    flops *= n
    if k == "film":
        # three forward and three inverse real transforms of the padded grid,
        # and the product with the symmetric tensor
        cells = 8.0 * n
        flops += evals * (6 * 2.5 * cells * math.log2(cells) + 36.0 * cells / 2)
    # each step reads and writes the spins once
    return {"bytes": 48.0 * n * case["steps"], "flops": flops * case["steps"]}


# ---------------------------------------------------------------------------
# the same from the equations, in 64-bit torch

def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _grid_index(size, periodic, nb, b, d, bb, offset, total, dev):
    """Index of the neighbour at cell + d, basis bb, for every cell of basis b
    (spin ((x Ly + y) Lz + z) nb + b, shifted by offset); `total` (a row of
    zeros) outside an open boundary."""
    ax = []
    ok = torch.ones((1, 1, 1), dtype=torch.bool, device=dev)
    for a in range(3):
        v = torch.arange(size[a], device=dev) + d[a]
        shape = [1, 1, 1]
        shape[a] = size[a]
        inside = (v >= 0) & (v < size[a])
        if not periodic:
            ok = ok & inside.view(shape)
        ax.append((v % size[a]).view(shape))
    idx = ((ax[0] * size[1] + ax[1]) * size[2] + ax[2]) * nb + bb + offset
    return torch.where(ok, idx, torch.full_like(idx, total)).reshape(-1)


def _stencil(rows, nb):
    """per basis site b: (cell offset, neighbour's basis site, 3x3 tensor)"""
    out = [[] for _ in range(nb)]
    for _, _, r, J in rows:
        J = np.asarray(J, np.float64).reshape(-1)
        T = float(J[0]) * np.eye(3) if J.size == 1 else J.reshape(3, 3)
        half = abs(r[0] - round(r[0])) > 0.25
        for b in range(nb):
            bb = 1 - b if half else b
            shift = 0.5 * (b - bb)
            out[b].append((tuple(int(round(x + shift)) for x in r), bb, T))
    return out


def _replica_size(case):
    """(lattice side, spins, basis sites) of each replica, from its description"""
    sides, ns, nbs = [], [], []
    for _, _, _, _, desc in configs.c4(case["n"]):
        side = int(desc.split()[1].split("^")[0])
        nb = 2 if desc.startswith("bcc") else 1
        sides.append(side)
        ns.append(nb * side ** 3)
        nbs.append(nb)
    return sides, ns, nbs


def _mulhilo(m, x):
    p = m * x                      # exact modulo 2^64
    return (p >> 32) & 0xFFFFFFFF, p & 0xFFFFFFFF


def _philox(c, k0, k1):
    """Philox4x32-10 (Salmon et al., SC'11) on int64 tensors holding 32-bit words"""
    for _ in range(10):
        hi0, lo0 = _mulhilo(0xD2511F53, c[0])
        hi1, lo1 = _mulhilo(0xCD9E8D57, c[2])
        c = (hi1 ^ c[1] ^ k0, lo1, hi0 ^ c[3] ^ k1, lo0)
        k0 = (k0 + 0x9E3779B9) & 0xFFFFFFFF
        k1 = (k1 + 0xBB67AE85) & 0xFFFFFFFF
    return c


def _normals(seed, step, spin):
    """The thermostat's three normals per spin: two Philox calls, Box-Muller."""
    def uniform(hi, lo):
        return ((hi << 20) | (lo >> 12)).double() * 2.0 ** -52 + 2.0 ** -53
    k0, k1 = seed & 0xFFFFFFFF, (seed >> 32) & 0xFFFFFFFF
    z = []
    for call in (0, 1):
        st = torch.full_like(spin, step)
        a = _philox((spin, torch.full_like(spin, call), st, torch.zeros_like(spin)), k0, k1)
        r = torch.sqrt(-2.0 * torch.log(uniform(a[0], a[1])))
        phi = 2.0 * math.pi * uniform(a[2], a[3])
        z += [r * torch.cos(phi), r * torch.sin(phi)]
    return torch.stack(z[:3], 1)


def _film_field(case, mus, dev):
    """h = mus sum_j mus W(r_ij) s_j over an open film, by zero-padded FFTs"""
    L = (case["x"], case["y"], case["z"])
    P = tuple(2 * v for v in L)
    r = []
    for a in range(3):
        n = torch.arange(P[a], device=dev, dtype=torch.float64)
        n = torch.where(n < L[a], n, n - P[a])
        shape = [1, 1, 1]
        shape[a] = P[a]
        r.append(n.view(shape).expand(P))
    r2 = r[0] ** 2 + r[1] ** 2 + r[2] ** 2
    far = r2 == 0
    for a in range(3):
        far = far | (r[a] == -L[a])
    pre = MU0 / (4.0 * math.pi * (0.3e-9) ** 3)
    inv5 = torch.where(far, torch.zeros_like(r2), r2.clamp(min=1.0) ** -2.5)
    W = {}
    for a in range(3):
        for b in range(a, 3):
            w = 3.0 * r[a] * r[b] - (r2 if a == b else 0.0)
            W[a, b] = W[b, a] = torch.fft.rfftn(pre * w * inv5)

    def field(s):
        S = [torch.fft.rfftn((mus * s[:, c]).view(L), s=P) for c in range(3)]
        h = [torch.fft.irfftn(sum(W[a, b] * S[b] for b in range(3)), s=P) for a in range(3)]
        return mus[:, None] * torch.stack([x[:L[0], :L[1], :L[2]].reshape(-1) for x in h], 1)
    return field


def exact(case, seed):
    dev = _device()
    k = case["kind"]
    f64 = dict(dtype=torch.float64, device=dev)
    K = field = None
    T = float(case.get("T", 0.0))
    # blocks of rows: (first, stride, [(neighbour index, coefficient)])
    blocks = []
    if k == "replicas":
        sides, ns, nbs = _replica_size(case)
        n = sum(ns)
        reps = _replicas(case, seed)
        off = np.concatenate([[0], np.cumsum(ns)])
        nbr = [torch.full((n,), n, dtype=torch.int64, device=dev) for _ in range(8)]
        for q, (side, nb) in enumerate(zip(sides, nbs)):
            st = _stencil(configs.sc_neighbour_rows(1.0) if nb == 1 else configs.bcc_nn_rows(1.0), nb)
            for b in range(nb):
                for m, (d, bb, _) in enumerate(st[b]):
                    nbr[m][off[q] + b:off[q + 1]:nb] = _grid_index((side,) * 3, True, nb, b, d, bb,
                                                                   int(off[q]), n, dev)
        blocks.append((0, 1, [(i, 1.0) for i in nbr]))
        moment, alpha, dt = 2.0, 0.1, 1e-3
        rep = torch.repeat_interleave(torch.arange(len(ns), device=dev), torch.tensor(ns, device=dev))
        T = torch.tensor([r[1] for r in reps], **f64)[rep][:, None]
        noise_seed = torch.tensor([r[2] for r in reps], device=dev)[rep]
        spin = torch.arange(n, device=dev) - torch.tensor(off[:-1], device=dev)[rep]
        mus = torch.full((n,), moment * BOHR, **f64)
        field = mus[:, None] * torch.tensor([r[3] for r in reps], **f64)[rep]
        alpha = torch.full((n,), alpha, **f64)
    elif k == "alloy":
        types, pi, pj = _alloy(case, seed)
        n = types.size
        m, _, al = _alloy_sites(types)
        mus, alpha, dt = torch.tensor(m, **f64), torch.tensor(al, **f64), 1e-3
        table = torch.tensor([[ALLOY_J[a, b] for b in (0, 1)] for a in (0, 1)], **f64)
        ty = torch.tensor(types, dtype=torch.int64, device=dev)
        ents = []
        for a, b in zip(pi, pj):
            idx = torch.full((n,), n, dtype=torch.int64, device=dev)
            idx[torch.tensor(a, dtype=torch.int64, device=dev)] = torch.tensor(b, dtype=torch.int64, device=dev)
            J = table[ty, torch.cat([ty, ty[:1]])[idx]]
            ents.append((idx, J[:, None]))
        blocks.append((0, 1, ents))
        noise_seed, spin = seed, torch.arange(n, device=dev)
    else:
        rows, nb, moment, al, dt, B, K = _material(case)
        size = (case["x"], case["y"], case["z"])
        n = nb * size[0] * size[1] * size[2]
        dt = dt / 1e-12
        mus = torch.full((n,), moment * BOHR, **f64)
        alpha = torch.full((n,), al, **f64)
        periodic = k != "film" and not case.get("open")
        for b, st in enumerate(_stencil(rows, nb)):
            ents = []
            for d, bb, J in st:
                iso = np.array_equal(J, J[0, 0] * np.eye(3))
                ents.append((_grid_index(size, periodic, nb, b, d, bb, 0, n, dev),
                             float(J[0, 0]) if iso else torch.tensor(J.T.copy(), **f64)))
            blocks.append((b, nb, ents))
        if B is not None:
            field = mus[:, None] * torch.tensor(B, **f64)[None, :]
        noise_seed, spin = seed, torch.arange(n, device=dev)
    dipole = _film_field(case, mus, dev) if k == "film" else None
    s = torch.tensor(_spins(n, seed), **f64)
    zero = torch.zeros((1, 3), **f64)

    def exchange(s):
        se = torch.cat([s, zero])
        h = torch.zeros_like(s)
        for first, stride, ents in blocks:
            acc = torch.zeros_like(s[first::stride])
            for idx, J in ents:
                g = se[idx]
                if isinstance(J, torch.Tensor) and J.shape == (3, 3):
                    acc = torch.addmm(acc, g, J)
                else:
                    acc = acc + J * g
            h[first::stride] = acc
        return h

    def rhs(s, w):
        h = exchange(s)
        if field is not None:
            h = h + field
        if K is not None:
            h[:, 2] += 2.0 * K * s[:, 2]
        if dipole is not None:
            h = h + dipole(s)
        h = h / mus[:, None] + w
        c = torch.linalg.cross(s, h)
        return -GYRO * (c + alpha[:, None] * torch.linalg.cross(s, c))

    def unit(v):
        return v / torch.linalg.vector_norm(v, dim=1, keepdim=True)

    sigma = torch.sqrt(2.0 * KB * alpha / (mus * GYRO * dt))[:, None]
    hot = k == "replicas" or T > 0.0
    for step in range(case["steps"]):
        w = _normals(noise_seed, step, spin) * sigma * T ** 0.5 if hot else 0.0
        if case.get("integrator") == "rk4":
            k1 = rhs(s, w)
            k2 = rhs(s + 0.5 * dt * k1, w)
            k3 = rhs(s + 0.5 * dt * k2, w)
            k4 = rhs(s + dt * k3, w)
            s = unit(s + dt * (k1 + 2.0 * k2 + 2.0 * k3 + k4) / 6.0)
        else:
            a = rhs(s, w)
            s = unit(s + 0.5 * dt * (a + rhs(unit(s + dt * a), w)))
    ms = torch.cat([mus[:, None] * s, mus[:, None]], 1)
    if k == "replicas":
        moments = torch.zeros((len(ns), 4), **f64).index_add_(0, rep, ms)
    else:
        moments = ms.sum(0)
    out = {"spins": s, "moments": moments}
    if k == "alloy":
        out["energy"] = (-0.5 * (s * exchange(s)).sum()).reshape(1)
    return out
