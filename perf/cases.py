"""The work this framework is used for, as cases that can be timed and compared.

A case is one whole call sequence of a user's program on a problem it already
holds: an anneal (random spins, a schedule of anneal_one_step calls, the
solution read back), an exhaustive search, a batch of anneals, or the energies
of a set of states.  Every case goes through the public entry points of
sqaod_amd.rocm with the defaults a user gets.

Couplings of the anneals and searches are integers in [-w, w], the law of
max-cut and number-partitioning style QUBOs: every local field and energy is
then exact in each float format, so one problem, seed and schedule has one
right trajectory and the outputs are compared bit by bit.  (On real-valued
couplings a last-bit difference in a single field, which any other order of
summation gives, sends the whole trajectory elsewhere.)  The energies of the
formulas are on N(0, 1) weights, against 64-bit sums.

The schedule is the usual one: G falls geometrically from 5 to 0.01, in 205
steps (a factor 0.97 each) where nothing else is said; beta = 50.
"""
import numpy as np
import torch

import sqaod_amd.rocm as rocm
from sqaod_amd.rocm import formulas

BETA = 50.0
STEPS = 205
_REAL = {"f32": np.float32, "f64": np.float64}


def _dense(name, n, m, dtype="f32", form="native", w=8, steps=STEPS):
    return {"name": name, "kind": "dense", "n": n, "m": m, "dtype": dtype, "form": form, "w": w, "steps": steps}


def _bipartite(name, n0, n1, m, dtype="f32", form="native", w=8, steps=STEPS):
    return {"name": name, "kind": "bipartite", "n0": n0, "n1": n1, "m": m, "dtype": dtype, "form": form, "w": w,
            "steps": steps}


def listed():
    return [
        # the smallest anneal in use: every step is launch and latency
        _dense("dense_n128_m32", 128, 32),
        # a mid-sized problem with everything left at its default: float64, n_trotters = N / 4
        _dense("dense_default_f64", 500, 125, dtype="f64"),
        # float32 at the default n_trotters of its size: more slices than the GPU has compute units
        _dense("dense_default_f32", 1200, 300),
        # the largest anneal: N=4096, m=256, couplings of about unit variance, J as bf16 hi + lo
        _dense("dense_n4096_bf16x2", 4096, 256, form="bf16x2", w=2),
        # simulated annealing: one replica, n_trotters = 1
        _dense("dense_sa_n1000", 1000, 1),
        # bipartite (RBM-shaped) problem of two equal layers
        _bipartite("bipartite_n1024_m64", 1024, 1024, 64),
        # two ragged layers with everything at its default: float64, n_trotters = (N0 + N1) / 4
        _bipartite("bipartite_default_f64", 200, 301, 125, dtype="f64"),
        # exhaustive search of a small problem at the default dtype: a ground state to check an anneal by
        {"name": "bf_n20_f64", "kind": "bf", "n": 20, "dtype": "f64", "w": 8},
        # exhaustive search of 2^30 states
        {"name": "bf_n30_f32", "kind": "bf", "n": 30, "dtype": "f32", "w": 8},
        # exhaustive search of 2^32 pairs
        {"name": "bipartite_bf_16x16", "kind": "bipartite_bf", "n0": 16, "n1": 16, "dtype": "f32", "w": 8},
        # many independent problems of mixed sizes annealed together
        {"name": "batch_64_bf16x2", "kind": "batch", "instances": 64, "nmin": 64, "nmax": 1024, "shapes": 7,
         "form": "bf16x2", "w": 8, "steps": 100},
        # energies of 500 given states under one QUBO
        {"name": "energies_n1000_b500", "kind": "energies", "graph": "dense", "n": 1000, "b": 500, "dtype": "f32"},
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["dense", "dense", "dense", "dense_f64", "sa", "bipartite", "bf", "bipartite_bf", "batch",
                       "energies"])
    if kind == "dense":
        n = _log_int(rng, 48, 3000)
        m = _log_int(rng, 4, max(4, min(256, n // 4)))
        return {k: v for k, v in _dense("", n, m, form=rng.choice(["native", "native", "bf16x2", "fp8"]),
                                        w=rng.choice([2, 8]), steps=rng.choice([100, 205])).items() if k != "name"}
    if kind == "dense_f64":
        n = _log_int(rng, 48, 700)
        return {k: v for k, v in _dense("", n, max(2, n // 4), dtype="f64", steps=100).items() if k != "name"}
    if kind == "sa":
        return {k: v for k, v in _dense("", _log_int(rng, 100, 2000), 1, dtype=rng.choice(["f32", "f64"]),
                                        steps=100).items() if k != "name"}
    if kind == "bipartite":
        dtype = rng.choice(["f32", "f32", "f64"])
        top = 1024 if dtype == "f32" else 400
        n0, n1 = _log_int(rng, 40, top), _log_int(rng, 40, top)
        return {k: v for k, v in _bipartite("", n0, n1, _log_int(rng, 8, 128), dtype=dtype,
                                            form=rng.choice(["native", "bf16x2"]) if dtype == "f32" else "native",
                                            w=rng.choice([2, 8]), steps=rng.choice([100, 205])).items()
                if k != "name"}
    if kind == "bf":
        return {"kind": "bf", "n": rng.randint(10, 29), "dtype": rng.choice(["f32", "f64"]),
                "w": rng.choice([2, 8])}
    if kind == "bipartite_bf":
        return {"kind": "bipartite_bf", "n0": rng.randint(6, 16), "n1": rng.randint(6, 15),
                "dtype": rng.choice(["f32", "f64"]), "w": 8}
    if kind == "batch":
        return {"kind": "batch", "instances": _log_int(rng, 8, 96), "nmin": 50, "nmax": _log_int(rng, 200, 1024),
                "shapes": rng.randint(1, 1 << 20), "form": rng.choice(["native", "bf16x2", "fp8"]), "w": 8,
                "steps": 50}
    if rng.random() < 0.5:
        return {"kind": "energies", "graph": "dense", "n": _log_int(rng, 20, 2000), "b": _log_int(rng, 1, 1000),
                "dtype": rng.choice(["f32", "f64"])}
    return {"kind": "energies", "graph": "bipartite", "n0": _log_int(rng, 20, 1000), "n1": _log_int(rng, 20, 1000),
            "b0": _log_int(rng, 1, 100), "b1": _log_int(rng, 1, 100), "dtype": rng.choice(["f32", "f64"])}


# ---------------------------------------------------------------- inputs

def _symmetric(u):
    return np.triu(u) + np.triu(u, 1).T


def _int_qubo(rng, n, w, real):
    return _symmetric(rng.integers(-w, w + 1, (n, n), dtype=np.int8)).astype(real)


def _int_bipartite(rng, n0, n1, w, real):
    return (rng.integers(-w, w + 1, n0).astype(real), rng.integers(-w, w + 1, n1).astype(real),
            rng.integers(-w, w + 1, (n1, n0)).astype(real))


def _batch_shapes(case):
    rng = np.random.default_rng(case["shapes"])
    ratio = case["nmax"] / case["nmin"]
    return [(int(round(case["nmin"] * ratio ** rng.random())), int(rng.choice([16, 32, 64, 128])))
            for _ in range(case["instances"])]


def _energy_inputs(case, seed):
    rng = np.random.default_rng(seed)
    real = _REAL[case["dtype"]]
    if case["graph"] == "dense":
        n = case["n"]
        return {"W": _symmetric(rng.standard_normal((n, n), dtype=np.float32)).astype(real),
                "x": rng.integers(0, 2, (case["b"], n), dtype=np.int8)}
    n0, n1 = case["n0"], case["n1"]
    return {"b0": rng.standard_normal(n0).astype(real), "b1": rng.standard_normal(n1).astype(real),
            "W": rng.standard_normal((n1, n0)).astype(real),
            "x0": rng.integers(0, 2, (case["b0"], n0), dtype=np.int8),
            "x1": rng.integers(0, 2, (case["b1"], n1), dtype=np.int8)}


def _schedule(steps):
    return [5.0 * (0.01 / 5.0) ** (k / (steps - 1)) for k in range(steps)]


def prepare(case, seed):
    kind, rng = case["kind"], np.random.default_rng(seed)
    if kind == "energies":
        return {"case": case, **_energy_inputs(case, seed)}
    if kind == "batch":
        solver = rocm.dense_batch(**({} if case["form"] == "native" else {"field_precision": case["form"]}))
        for i, (n, m) in enumerate(_batch_shapes(case)):
            solver.add_qubo(_int_qubo(rng, n, case["w"], np.float32), m, seed + i)
        solver.prepare()
        return {"case": case, "solver": solver, "G": np.array(_schedule(case["steps"]))}
    real = _REAL[case["dtype"]]
    if kind == "bf":
        return {"case": case, "solver": rocm.dense_graph_bf_searcher(_int_qubo(rng, case["n"], case["w"], real),
                                                                     dtype=real)}
    if kind == "bipartite_bf":
        problem = _int_bipartite(rng, case["n0"], case["n1"], case["w"], real)
        return {"case": case, "solver": rocm.bipartite_graph_bf_searcher(*problem, dtype=real)}
    prefs = {"n_trotters": case["m"]}
    if case["form"] != "native":
        prefs["field_precision"] = case["form"]
    if kind == "dense":
        solver = rocm.dense_graph_annealer(_int_qubo(rng, case["n"], case["w"], real), dtype=real, **prefs)
    else:
        problem = _int_bipartite(rng, case["n0"], case["n1"], case["w"], real)
        solver = rocm.bipartite_graph_annealer(*problem, dtype=real, **prefs)
    solver.seed(seed)
    solver.prepare()
    return {"case": case, "solver": solver, "G": _schedule(case["steps"])}


# ---------------------------------------------------------------- one pass

def _rows(x):
    """A solver's solutions (a list of rows, or of pairs of rows) as arrays."""
    if len(x) and isinstance(x[0], tuple):
        return [np.stack([a for a, _ in x]), np.stack([b for _, b in x])]
    return np.stack(x)


def _listed_solutions(case, x):
    """A search's solutions, -1 after the last: as many rows as a searcher
    lists at most (1024, or N0 + N1 pairs)."""
    if case["kind"] == "bf":
        x = [np.asarray(r) for r in x]
        width, most = case["n"], 1024
    else:
        x = [np.concatenate(r) for r in x]
        width = most = case["n0"] + case["n1"]
    out = np.full((most, width), -1, np.int8)
    out[:len(x)] = np.stack(x)
    return out


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "energies":
        real = _REAL[case["dtype"]]
        if case["graph"] == "dense":
            return formulas.dense_graph_batch_calculate_E(state["W"], state["x"], real)
        return formulas.bipartite_graph_batch_calculate_E_2d(state["b0"], state["b1"], state["W"], state["x0"],
                                                             state["x1"], real)
    solver = state["solver"]
    if kind == "batch":
        solver.prepare()
        solver.anneal(state["G"], BETA)
        n = len(solver)
        return {"E": np.concatenate([solver.get_E(i) for i in range(n)]),
                "x": np.concatenate([np.concatenate([np.ravel(r) for r in solver.get_x(i)]) for i in range(n)])}
    if kind in ("bf", "bipartite_bf"):
        solver.search()
        return {"E": solver.get_E()[:1], "x": _listed_solutions(case, solver.get_x())}
    solver.randomize_spin()
    for G in state["G"]:
        solver.anneal_one_step(G, BETA)
    solver.make_solution()
    return {"E": solver.get_E(), "x": _rows(solver.get_x())}


# ---------------------------------------------------------------- what a pass cannot do without

def _size(case):
    return 4 if case.get("dtype", "f32") == "f32" else 8


def work(case):
    """Bytes: the couplings and states once in, the results once out.  Flops:
    an anneal forms every slice's fields and energies once (2 m N^2 each) and
    about 20 operations an attempt; the fields' changes by accepted flips depend
    on the data and are left out.  A search adds and compares once a state."""
    kind, s = case["kind"], _size(case)
    if kind == "energies":
        if case["graph"] == "dense":
            n, b = case["n"], case["b"]
            return {"bytes": s * n * n + b * n + s * b, "flops": 2.0 * b * n * n}
        n0, n1, b0, b1 = case["n0"], case["n1"], case["b0"], case["b1"]
        return {"bytes": s * (n0 * n1 + n0 + n1 + b0 * b1) + b0 * n0 + b1 * n1,
                "flops": 2.0 * b0 * n0 * n1 + 2.0 * b0 * b1 * n1}
    if kind == "bf":
        return {"bytes": s * case["n"] ** 2 + case["n"] + s, "flops": 2.0 * 2 ** case["n"]}
    if kind == "bipartite_bf":
        n0, n1 = case["n0"], case["n1"]
        return {"bytes": s * (n0 * n1 + n0 + n1) + n0 + n1 + s, "flops": 2.0 * 2 ** (n0 + n1)}
    if kind == "batch":
        shapes, steps = _batch_shapes(case), case["steps"]
        return {"bytes": float(sum(4 * n * n + n * m + 4 * m for n, m in shapes)),
                "flops": float(sum(4 * m * n * n + 20 * steps * m * n for n, m in shapes))}
    m, steps = case["m"], case["steps"]
    if kind == "dense":
        n = case["n"]
        return {"bytes": s * n * n + m * n + s * m, "flops": 4.0 * m * n * n + 20.0 * steps * m * n}
    # a bipartite step forms both layers' fields anew: its flips are decided a layer at a time
    n0, n1 = case["n0"], case["n1"]
    return {"bytes": s * n0 * n1 + m * (n0 + n1) + s * m,
            "flops": 4.0 * steps * m * n0 * n1 + 20.0 * steps * m * (n0 + n1)}


def tolerance(case):
    if case["kind"] != "energies":
        return "exact"
    # sums in 64 bits and one rounding to the result's type
    return {"rel": 1e-7, "max": 5e-7} if case["dtype"] == "f32" else {"rel": 1e-13, "max": 1e-12}


# ---------------------------------------------------------------- the same in plain 64 bits

def _bits(lo, hi, n, device):
    """Rows x = lo .. hi-1 as n float64 bits, the highest first."""
    x = torch.arange(lo, hi, device=device)
    return ((x[:, None] >> torch.arange(n - 1, -1, -1, device=device)) & 1).double()


def _minimum(row_energies, rows, chunk):
    """The least energy over blocks of rows."""
    return min(float(row_energies(lo, min(rows, lo + chunk)).min()) for lo in range(0, rows, chunk))


def exact(case, seed):
    kind = case["kind"]
    if kind == "energies":
        v = {k: a.astype(np.float64) for k, a in _energy_inputs(case, seed).items()}
        if case["graph"] == "dense":
            return np.sum((v["x"] @ v["W"]) * v["x"], axis=1)
        return (v["x1"] @ v["W"] @ v["x0"].T + (v["x0"] @ v["b0"])[None, :] + (v["x1"] @ v["b1"])[:, None])
    if kind not in ("bf", "bipartite_bf"):
        return None  # the end of a random walk: no value of its own in plain torch
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    rng = np.random.default_rng(seed)
    if kind == "bf":
        n = case["n"]
        W = torch.tensor(_int_qubo(rng, n, case["w"], np.float64), device=dev)
        low = min(n, 14)
        high = n - low
        xl = _bits(0, 1 << low, low, dev)
        el = ((xl @ W[high:, high:]) * xl).sum(1)

        def row_energies(lo, hi):
            xh = _bits(lo, hi, high, dev)
            return ((xh @ W[:high, :high]) * xh).sum(1)[:, None] + el[None, :] + 2.0 * ((xh @ W[:high, high:]) @ xl.T)

        rows = 1 << high
    else:
        n0, n1 = case["n0"], case["n1"]
        b0, b1, W = (torch.tensor(a, device=dev) for a in _int_bipartite(rng, n0, n1, case["w"], np.float64))
        x0 = _bits(0, 1 << n0, n0, dev)
        e0 = x0 @ b0

        def row_energies(lo, hi):
            x1 = _bits(lo, hi, n1, dev)
            return (x1 @ W) @ x0.T + e0[None, :] + (x1 @ b1)[:, None]

        rows = 1 << n1
    return {"E": np.array([_minimum(row_energies, rows, 4096)]), "x": None}
