"""What the engine is timed on: calls that users of the package make.

Each case is one call through a public entry point (``Solver``, the torch RBM
step, ``Problem.energy``, or the C entry points that take device pointers, as
INTEGRATION.md describes them), at the sizes of this repository's benchmark
configurations and tests.  ``prepare`` makes the problem and what a program
keeps beside it; ``run`` is one call on it.  Every run passes a seed, so that
two passes over the same state give the same chains.
"""

import math

import numpy as np
import torch  # before the engine library is loaded: both then share one HIP runtime

from pysa_amd import _lib, batched, instances
from pysa_amd.sa import Solver
from pysa_amd.torch_rbm import update_states_with_pysa

# device-resident runs (see "Keeping inputs in device memory" in INTEGRATION.md)
_FORMS = {"plain": (_lib.FORM_PLAIN, "random"), "blocked": (_lib.FORM_BLOCKED, "block_random"),
          "blocked_exact": (_lib.FORM_BLOCKED_EXACT, "block_random")}


def listed():
    return [
        # The smallest calls: a tuning loop (TTS, ladder search) over a 50-spin
        # instance, a handful of short reads, energies recomputed in f64 to
        # judge success.  PySA's default random order.
        dict(name="small_n50", kind="solver", problem="pm1", n=50, reads=10, replicas=4,
             sweeps=100, strategy="random", dtype="float32", tmin=0.3, tmax=1.5,
             recompute=True),
        # Dense +-1 Ising, 64 spins, many reads, sequential order.
        dict(name="pm1_n64", kind="solver", problem="pm1", n=64, reads=32, replicas=16,
             sweeps=1000, strategy="sequential", dtype="float32", tmin=1.0, tmax=3.5),
        # Partition function of a 16x16 +-1 lattice with local fields: log Z from the
        # exchange ladder (get_part_fun), outputs sorted by temperature.
        dict(name="lattice_logz", kind="solver", problem="lattice", n=256, reads=16, replicas=32,
             sweeps=1000, strategy="sequential", dtype="float32", tmin=0.5, tmax=3.0,
             part_fun=True),
        # float64 problems: an ordinary PT run in double precision.
        dict(name="gauss_f64_n300", kind="solver", problem="gauss", n=300, reads=8, replicas=16,
             sweeps=100, strategy="random", dtype="float64", tmin=0.5, tmax=5.0),
        # Dense QUBO with Gaussian couplings, the default random order.
        dict(name="qubo_n512", kind="solver", problem="qubo", n=512, reads=128, replicas=32,
             sweeps=1000, strategy="random", dtype="float32", tmin=0.1, tmax=5.0),
        # PySA's own timing of one big instance: 3072 spins, 100 replicas, one
        # read, sequential order, no exchanges.
        dict(name="ising_n3072", kind="solver", problem="gauss", n=3072, reads=1, replicas=100,
             sweeps=2, strategy="sequential", dtype="float32", tmin=5.0, tmax=50.0,
             use_pt=False),
        # Planted Wishart instance, 1024 spins, resident in HBM: the production
        # batch in the MFMA form (the largest case) and in the plain form.
        dict(name="wishart_n1024", kind="resident", form="blocked", n=1024, reads=512,
             replicas=32, sweeps=1000, tmin=0.3, tmax=1.5),
        dict(name="wishart_n1024_plain", kind="resident", form="plain", n=1024, reads=512,
             replicas=32, sweeps=40, tmin=0.3, tmax=1.5),
        # Negative phase of RBM training on device tensors, 784 + 500 units.
        dict(name="rbm_step", kind="rbm", visible=784, hidden=500, chains=64, steps=5),
        # Annealed importance sampling of an RBM-shaped Ising model.
        dict(name="ais_n1284", kind="ais", visible=784, hidden=500, chains=2048, temps=500,
             reference="uniform"),
        # Many Sherrington-Kirkpatrick instances of uneven size in one call.
        dict(name="sk_batch", kind="batch", count=256, nmin=32, nmax=768, reads=4, replicas=8,
             sweeps=500),
        # f64 energies of a batch of states (success tests after a run).
        dict(name="energy_n1024", kind="energy", n=1024, count=16384, dtype="float32"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["solver", "solver", "solver", "resident", "rbm", "ais", "batch", "energy"])
    if kind == "solver":
        flavour = rng.choice(["small", "float64", "mfma", "mfma", "large"])
        strategy = rng.choice(["random", "sequential"])
        c = dict(kind=kind, strategy=strategy, dtype="float32",
                 reads=_log_int(rng, 1, 64), replicas=_log_int(rng, 2, 64))
        if flavour == "small":  # tuning loops: small instances, short reads
            c.update(problem="pm1", n=rng.randint(12, 64), sweeps=_log_int(rng, 50, 1000),
                     tmin=0.3, tmax=2.0, recompute=rng.random() < 0.5)
        elif flavour == "float64":
            c.update(problem=rng.choice(["gauss", "qubo"]), dtype="float64",
                     n=_log_int(rng, 20, 700), reads=_log_int(rng, 1, 32), replicas=_log_int(rng, 2, 32),
                     sweeps=_log_int(rng, 10, 60), tmin=0.5, tmax=5.0)
        elif flavour == "mfma":  # what form='auto' runs on the matrix cores
            c.update(problem=rng.choice(["gauss", "qubo", "pm1", "wishart"]),
                     n=_log_int(rng, 65, 1100), sweeps=_log_int(rng, 50, 500), tmin=0.3, tmax=5.0)
        else:  # one big instance, one read, many replicas
            c.update(problem="gauss", n=_log_int(rng, 2049, 3300), reads=1,
                     replicas=_log_int(rng, 8, 128), sweeps=rng.randint(1, 3),
                     tmin=5.0, tmax=50.0, use_pt=rng.random() < 0.5)
        return c
    if kind == "resident":
        form = rng.choice(["blocked", "blocked_exact", "plain"])
        n = _log_int(rng, 200, 1024)
        return dict(kind=kind, form=form, n=n, reads=_log_int(rng, 32, 512),
                    replicas=rng.choice([8, 16, 32]), sweeps=20 if form == "plain" else 300,
                    tmin=0.3, tmax=1.5)
    if kind == "rbm":
        return dict(kind=kind, visible=_log_int(rng, 50, 784), hidden=_log_int(rng, 20, 500),
                    chains=_log_int(rng, 8, 128), steps=rng.randint(1, 10))
    if kind == "ais":
        ref = rng.choice(["uniform", "uniform", "bernoulli"])
        return dict(kind=kind, visible=_log_int(rng, 40, 784), hidden=_log_int(rng, 30, 500),
                    chains=_log_int(rng, 64, 2048) if ref == "uniform" else _log_int(rng, 64, 1024),
                    temps=_log_int(rng, 50, 500) if ref == "uniform" else _log_int(rng, 20, 100),
                    reference=ref)
    if kind == "batch":
        nmin = _log_int(rng, 20, 200)
        return dict(kind=kind, count=_log_int(rng, 8, 256), nmin=nmin,
                    nmax=nmin + rng.randint(1, 500), reads=rng.randint(1, 6),
                    replicas=rng.choice([4, 8, 16]), sweeps=_log_int(rng, 50, 500))
    return dict(kind="energy", n=_log_int(rng, 50, 3072), count=_log_int(rng, 1, 16384),
                dtype=rng.choice(["float32", "float64"]))


# ------------------------------------------------------------------ problems --
def _symmetric(a):
    a = np.triu(a, 1)
    return a + a.T


def _problem(kind, n, rng):
    """A problem in PySA's convention (diagonal: local fields)."""
    if kind == "pm1":
        return _symmetric(2.0 * rng.integers(0, 2, (n, n)) - 1)
    if kind == "gauss":
        return _symmetric(rng.standard_normal((n, n))) + np.diag(rng.standard_normal(n))
    if kind == "qubo":
        return instances.gaussian_qubo(n, int(rng.integers(2**31))).astype(np.float64)
    if kind == "wishart":
        return instances.planted_wishart(n, 0.5, int(rng.integers(2**31)))[0].astype(np.float64)
    side = int(round(math.sqrt(n)))  # periodic lattice, small integer local fields
    p = np.zeros((n, n))
    for i in range(side):
        for j in range(side):
            for k in (((i + 1) % side) * side + j, i * side + (j + 1) % side):
                p[i * side + j, k] = p[k, i * side + j] = 2 * rng.integers(0, 2) - 1
    return p + np.diag(rng.integers(-1, 2, n).astype(np.float64))


def _energy_inputs(case, seed):
    rng = np.random.default_rng([seed, 7])
    n = case["n"]
    p = _symmetric(rng.standard_normal((n, n), dtype=np.float32))
    h = rng.standard_normal(n, dtype=np.float32)
    s = (2 * rng.integers(0, 2, (case["count"], n), dtype=np.int8) - 1).astype(np.int8)
    return p, h, s


# ------------------------------------------------------------------- prepare --
def prepare(case, seed):
    rng = np.random.default_rng([seed, 1])
    kind = case["kind"]
    if kind == "solver":
        ptype = "qubo" if case["problem"] == "qubo" else "ising"
        p = _problem(case["problem"], case["n"], rng)
        return dict(case=case, seed=seed, solver=Solver(p, ptype, float_type=case["dtype"]))
    if kind == "resident":
        return _prepare_resident(case, seed, rng)
    if kind == "rbm":
        g = torch.Generator().manual_seed(seed)
        nv, nh, r = case["visible"], case["hidden"], case["chains"]
        t = dict(W=0.05 * torch.randn(nv, nh, generator=g),
                 v_bias=0.1 * torch.randn(nv, 1, generator=g),
                 h_bias=0.1 * torch.randn(nh, 1, generator=g),
                 v_state=torch.randint(0, 2, (r, nv), generator=g).float(),
                 h_state=torch.randint(0, 2, (r, nh), generator=g).float())
        return dict(case=case, seed=seed, **{k: v.cuda() for k, v in t.items()})
    if kind == "ais":
        p = instances.rbm_ising(case["visible"], case["hidden"], seed=seed)
        return dict(case=case, seed=seed, solver=Solver(p, "ising"))
    if kind == "batch":
        return _prepare_batch(case, seed, rng)
    p, h, s = _energy_inputs(case, seed)
    return dict(case=case, states=s,
                problem=_lib.Problem(p, h, "ising", np.dtype(case["dtype"])))


def _ladder(replicas, tmin, tmax):
    if replicas == 1:
        return np.array([1 / tmin], dtype=np.float32)
    return (1 / np.geomspace(tmin, tmax, replicas)).astype(np.float32)


def _prepare_resident(case, seed, rng):
    n, reads, r = case["n"], case["reads"], case["replicas"]
    p, _ = instances.planted_wishart(n, 0.5, int(rng.integers(2**31)))
    h = np.zeros(n, np.float32)
    prob = _lib.Problem(p, h, "ising", np.float32)
    states = (2 * rng.integers(0, 2, (reads, r, n), dtype=np.int8) - 1).astype(np.int8)
    sd = torch.from_numpy(states).cuda()
    x = sd.reshape(-1, n).double()
    energies = (0.5 * ((x @ torch.from_numpy(p).cuda().double()) * x).sum(1)).float()
    betas = _ladder(r, case["tmin"], case["tmax"])
    order = np.argsort(betas, kind="quicksort").astype(np.int32)
    out = dict(states=torch.empty_like(sd), energies=torch.empty_like(energies).reshape(reads, r),
               beta_idx=torch.empty((reads, r), dtype=torch.int64, device="cuda"),
               best_state=torch.empty((reads, n), dtype=torch.int8, device="cuda"),
               best_energy=torch.empty(reads, dtype=torch.float32, device="cuda"),
               best_sweeps=torch.empty(reads, dtype=torch.int32, device="cuda"),
               accepted=torch.empty(reads, dtype=torch.int64, device="cuda"))
    return dict(case=case, seed=seed, problem=prob, stream=torch.cuda.Stream(), states0=sd,
                energies0=energies.reshape(reads, r), betas=torch.from_numpy(betas).cuda(),
                order=torch.from_numpy(order).cuda(), out=out)


def _prepare_batch(case, seed, rng):
    reads, r, count = case["reads"], case["replicas"], case["count"]
    # the sizes belong to the case, the couplings and states to the seed
    sizes = np.random.default_rng([count, case["nmin"], case["nmax"]])
    inst = []
    for _ in range(count):
        n = int(sizes.integers(case["nmin"], case["nmax"] + 1))
        a = np.triu(2 * rng.integers(0, 2, (n, n), dtype=np.int8) - 1, 1)
        inst.append((a + a.T, np.float32(1 / math.sqrt(n))))
    pk = batched.pack(inst)
    ns = pk["n"].astype(np.int64)
    total = int(reads * r * ns.sum())
    states = (2 * rng.integers(0, 2, total, dtype=np.int8) - 1).astype(np.int8)
    s_off = np.concatenate([[0], np.cumsum(reads * r * ns)[:-1]]).astype(np.int64)
    dev = {k: torch.from_numpy(np.ascontiguousarray(v)).cuda() for k, v in pk.items()}
    sd = torch.from_numpy(states).cuda()
    en = []
    for (s, scale), o, n in zip(inst, s_off, ns):
        x = sd[int(o):int(o) + reads * r * int(n)].reshape(reads * r, int(n)).float()
        f = x @ torch.from_numpy(s).cuda().float()  # whole numbers, exact
        en.append(((f * x).sum(1).double() * (0.5 * float(scale))).float())
    energies = torch.cat(en).reshape(count * reads, r)
    betas = torch.from_numpy(np.tile(_ladder(r, 0.3, 1.5), (count, 1))).cuda()
    out = dict(states=torch.empty_like(sd), energies=torch.empty_like(energies),
               beta_idx=torch.empty((count * reads, r), dtype=torch.int64, device="cuda"),
               best_state=torch.empty(total // r, dtype=torch.int8, device="cuda"),
               best_energy=torch.empty(count * reads, dtype=torch.float32, device="cuda"),
               best_sweeps=torch.empty(count * reads, dtype=torch.int32, device="cuda"),
               accepted=torch.empty(count * reads, dtype=torch.int64, device="cuda"))
    return dict(case=case, seed=seed, stream=torch.cuda.Stream(), dev=dev, states0=sd,
                energies0=energies, betas=betas, s_off=torch.from_numpy(s_off).cuda(), out=out)


# ----------------------------------------------------------------------- run --
def run(state):
    return {"solver": _run_solver, "resident": _run_resident, "rbm": _run_rbm, "ais": _run_ais,
            "batch": _run_batch, "energy": _run_energy}[state["case"]["kind"]](state)


def _run_solver(state):
    c = state["case"]
    np.random.seed(state["seed"] % 2**32)  # the initial states come from NumPy's global RNG
    res = state["solver"].metropolis_update(
        num_sweeps=c["sweeps"], num_reads=c["reads"], num_replicas=c["replicas"],
        min_temp=c["tmin"], max_temp=c["tmax"], update_strategy=c["strategy"],
        recompute_energy=c.get("recompute", False), use_pt=c.get("use_pt", True),
        get_part_fun=c.get("part_fun", False), sort_output_temps=c.get("part_fun", False),
        return_dataframe=False, seed=state["seed"])
    keys = ["states", "energies", "best_state", "best_energy", "temps", "min_sweeps"]
    if c.get("part_fun", False):
        keys.append("log_Zf")
    return {k: np.array([r[k] for r in res]) for k in keys}


def _run_resident(state):
    c, o = state["case"], state["out"]
    form, order = _FORMS[c["form"]]
    stream = state["stream"]
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        o["states"].copy_(state["states0"])
        o["energies"].copy_(state["energies0"])
        _lib.check(_lib.load().pysa_amd_metropolis_device(
            state["problem"].handle, c["reads"], c["replicas"], c["sweeps"], _lib.ORDER[order], 1,
            0, 0, state["betas"].data_ptr(), state["order"].data_ptr(), state["seed"], 0, form, 0,
            None, None, None, o["states"].data_ptr(), o["energies"].data_ptr(),
            o["beta_idx"].data_ptr(), o["best_state"].data_ptr(), o["best_energy"].data_ptr(),
            o["best_sweeps"].data_ptr(), None, o["accepted"].data_ptr(), None,
            stream.cuda_stream))
    return o


def _run_rbm(state):
    v, h = update_states_with_pysa(state["W"], state["v_bias"], state["h_bias"], state["v_state"],
                                   state["h_state"], state["case"]["steps"], min_temp=1.0,
                                   max_temp=3.5, seed=state["seed"])
    return dict(v_state=v, h_state=h)


def _run_ais(state):
    c = state["case"]
    np.random.seed(state["seed"] % 2**32)
    logz, samples, omegas = state["solver"].annealed_importance(
        c["temps"], c["chains"], c["reference"], seed=state["seed"],
        reference_args=[0.4] if c["reference"] == "bernoulli" else None)
    return dict(logZf=float(logz), samples=samples, omegas=np.array(omegas))


def _run_batch(state):
    c, o, d = state["case"], state["out"], state["dev"]
    stream = state["stream"]
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        o["states"].copy_(state["states0"])
        o["energies"].copy_(state["energies0"])
        _lib.check(_lib.load().pysa_amd_batched_device(
            c["count"], d["n"].data_ptr(), d["ld"].data_ptr(), d["j_off"].data_ptr(),
            d["signs"].data_ptr(), d["scale"].data_ptr(), None, None, 0, c["reads"],
            c["replicas"], c["sweeps"], _lib.ORDER["block_random"], 1, 0, state["betas"].data_ptr(),
            state["seed"], 0, state["s_off"].data_ptr(), o["states"].data_ptr(),
            o["energies"].data_ptr(), o["beta_idx"].data_ptr(), o["best_state"].data_ptr(),
            o["best_energy"].data_ptr(), o["best_sweeps"].data_ptr(), o["accepted"].data_ptr(),
            _lib.FORM_AUTO, None, stream.cuda_stream))
    return o


def _run_energy(state):
    return dict(energies=state["problem"].energy(state["states"]))


# ---------------------------------------------------------------- accounting --
def work(case):
    """A spin update needs its local field: 2 n flop, as in the reference's row
    product.  Bytes: couplings, fields and states in, states and best states
    out, once each."""
    kind = case["kind"]
    if kind == "batch":
        mean = (case["nmin"] + case["nmax"]) / 2
        sq = mean**2 + (case["nmax"] - case["nmin"])**2 / 12
        chains = case["reads"] * case["replicas"]
        return {"bytes": case["count"] * (sq + (2 * chains + case["reads"]) * mean),
                "flops": 2.0 * case["count"] * sq * chains * case["sweeps"]}
    if kind == "energy":
        n, count = case["n"], case["count"]
        size = np.dtype(case["dtype"]).itemsize
        return {"bytes": size * n * (n + 1) + count * (n + 8), "flops": 2.0 * n * n * count}
    if kind == "rbm":
        n, chains, sweeps = case["visible"] + case["hidden"], case["chains"], case["steps"]
        return {"bytes": 4.0 * case["visible"] * case["hidden"] + 8.0 * n * chains,
                "flops": 2.0 * n * n * chains * sweeps}
    if kind == "ais":
        n, chains, sweeps = case["visible"] + case["hidden"], case["chains"], case["temps"]
        return {"bytes": 4.0 * n * (n + 1) + 2.0 * n * chains,
                "flops": 2.0 * n * n * chains * sweeps}
    n, chains = case["n"], case["reads"] * case["replicas"]
    size = 8 if case.get("dtype") == "float64" else 4
    return {"bytes": size * n * (n + 1) + n * (2.0 * chains + case["reads"]),
            "flops": 2.0 * n * n * chains * case["sweeps"]}


def exact(case, seed):
    """f64 energies of given states.  The other cases return Monte Carlo
    chains: their numbers belong to the states that the engine's own random
    stream leads to, so there is no value to give beside it."""
    if case["kind"] != "energy":
        return None
    p, h, s = _energy_inputs(case, seed)
    p, h = p.astype(np.float64), h.astype(np.float64)
    out = np.empty(len(s))
    for k in range(0, len(s), 2048):
        x = s[k:k + 2048].astype(np.float64)
        out[k:k + 2048] = 0.5 * np.einsum("ij,ij->i", x @ p, x) + x @ h
    return dict(energies=out)
