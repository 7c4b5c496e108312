"""The calls whose speed is measured, over the sizes and options this framework is used at.

Every case is one pass of a user's program through the public entry points: `run_dynamics` for the small
ensembles that are called often, and for the production ensembles the `Ensemble` handle that such a program
keeps, with its problem, model and initial conditions loaded, and reads reductions and fields from after
each run.  The models, step sizes and distributions are those of the repository's benchmark and tests.
"""
import functools
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "nqcdynamics.jl_amd"))

import nqcd_mi355x as NQ  # noqa: E402
from nqcd_mi355x import _lib as L  # noqa: E402

MASS = 2000.0
TULLY = {1: [0.01, 1.6, 0.005, 1.0], 2: [0.1, 0.28, 0.015, 0.06, 0.05], 3: [6e-4, 0.1, 0.9]}
TULLY_MODEL = {1: NQ.TullyModelOne, 2: NQ.TullyModelTwo, 3: NQ.TullyModelThree}
MORSE3_FSSH = [0.02, 0.4, 4.0, 0.02, 0.02, 0.65, 4.5, 0.0, 0.003, 0.65, 6.0, 0.02,
               0.005, 32.0, 3.40, 0.0, 32.0, 4.8, 0.005, 32.0, 4.97]
MORSE3_MAP = [0.02, 0.5, 4.0, 0.0, 0.02, 0.5, 4.0, 0.004, 0.02, 0.5, 4.0, 0.008,
              0.003, 0.5, 4.0, 0.002, 0.5, 4.2, 0.003, 0.5, 4.4]
WELL = [1 / 1200, 1 / 40, 0.01, 0.005, 1.0]
RP_MASS, RP_BETA = 1836.0, 8.0
DIATOM_MASS = [12859.0, 12859.0]
IESH_GAMMA = 6.4e-3


def listed():
    return [
        # an interactive call: a few hundred trajectories for a few hundred steps, everything from opening
        # the device to the means, as a user's script or a parameter scan makes it over and over
        {"name": "call_fssh_small", "path": "call", "method": "fssh", "model": 1, "ntraj": 200, "nsteps": 800,
         "save_every": 200},
        # production FSSH: 1e6 trajectories mixing the three Tully models on a momentum grid, uneven lengths
        {"name": "mixed_fssh_1e6", "path": "mixed", "ntraj": 1_000_000, "precision": "fp32"},
        # mean-field dynamics in FP64 with populations and energies on a time grid and the final states kept
        {"name": "ehrenfest_fp64", "path": "two_state", "method": "ehrenfest", "model": 2, "ntraj": 100_000,
         "nsteps": 1000, "save_every": 50},
        # an open system: two states in a bath of 100 modes, population correlation function
        {"name": "spin_boson_fssh", "path": "spin_boson", "method": "fssh", "ntraj": 100_000, "nsteps": 1000},
        # quantum nuclei: ring polymers on one surface, and hopping between two
        {"name": "rpmd_p32", "path": "rpmd", "beads": 32, "ntraj": 100_000, "nsteps": 1000},
        {"name": "rpsh_p8", "path": "rpsh", "beads": 8, "ntraj": 100_000, "nsteps": 1000},
        # the learned Hamiltonian in the trajectories, and its training
        {"name": "surrogate_fssh", "path": "diatom", "surrogate": True, "ntraj": 200_000, "nsteps": 3000},
        {"name": "surrogate_train", "path": "train", "samples": 131072, "steps": 1000, "batch": 2048},
        # molecules at metals: independent electrons in 40 and in 100 discretised states
        {"name": "iesh_41_states", "path": "iesh", "method": "iesh", "levels": 40, "ntraj": 8192, "nsteps": 100},
        {"name": "iesh_101_states", "path": "iesh", "method": "iesh", "levels": 100, "ntraj": 2048, "nsteps": 50},
        # more than two states: photodissociation by hopping, and the mapping form of the same size
        {"name": "morse3_fssh", "path": "morse", "ntraj": 100_000, "nsteps": 1000, "precision": "fp32"},
        {"name": "spin_mapping_3", "path": "mapping", "method": "spin", "nstates": 3, "ntraj": 500_000, "nsteps": 500},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(["call", "mixed", "two_state", "spin_boson", "rpmd", "rpsh", "diatom", "train", "iesh", "morse",
                       "mapping"])
    if path == "call":
        steps = _log(rng, 100, 2000)
        return {"path": path, "method": rng.choice(["fssh", "ehrenfest"]), "model": rng.choice([1, 2, 3]),
                "ntraj": _log(rng, 64, 4096), "nsteps": steps, "save_every": max(1, steps // rng.choice([1, 3, 10]))}
    if path == "mixed":
        return {"path": path, "ntraj": _log(rng, 3000, 1_000_000), "precision": rng.choice(["fp32", "fp64"])}
    if path == "two_state":
        steps = _log(rng, 200, 1000)
        return {"path": path, "method": rng.choice(["ehrenfest", "fssh"]), "model": rng.choice([1, 2, 3]),
                "ntraj": _log(rng, 1000, 100_000), "nsteps": steps, "save_every": max(1, steps // rng.choice([5, 10, 20]))}
    if path == "spin_boson":
        return {"path": path, "method": rng.choice(["fssh", "ehrenfest"]), "ntraj": _log(rng, 1000, 100_000),
                "nsteps": _log(rng, 200, 1000)}
    if path in ("rpmd", "rpsh"):
        beads = rng.choice([4, 8, 16, 32]) if path == "rpmd" else rng.choice([4, 8, 16])
        return {"path": path, "beads": beads, "ntraj": _log(rng, 1000, 100_000), "nsteps": _log(rng, 200, 1000)}
    if path == "diatom":
        return {"path": path, "surrogate": rng.random() < 0.6, "ntraj": _log(rng, 4000, 200_000),
                "nsteps": _log(rng, 500, 3000)}
    if path == "train":
        return {"path": path, "samples": _log(rng, 5000, 131072), "steps": _log(rng, 100, 1000),
                "batch": rng.choice([256, 1000, 1024, 2048])}
    if path == "iesh":
        levels = rng.randint(20, 100)
        most = 8192 if levels <= 50 else 2048
        return {"path": path, "method": rng.choice(["iesh", "iesh", "ehrenfest_na"]), "levels": levels,
                "ntraj": _log(rng, 200, most), "nsteps": _log(rng, 20, 50)}
    if path == "morse":
        return {"path": path, "ntraj": _log(rng, 1000, 100_000), "nsteps": _log(rng, 200, 1000),
                "precision": rng.choice(["fp32", "fp64"])}
    return {"path": path, "method": rng.choice(["spin", "ecmm"]), "nstates": rng.choice([2, 3]),
            "ntraj": _log(rng, 3000, 500_000), "nsteps": _log(rng, 100, 500)}


# --- inputs ---------------------------------------------------------------------------------------
def _rng(case, seed):
    return np.random.default_rng([int(seed), 77])


def _two_state_initial(case, seed):
    """(r0, v0) of a wave packet coming from the left: momentum 10 to 30 a.u., and the pure lower state."""
    rng, n = _rng(case, seed), case["ntraj"]
    p = rng.uniform(10.0, 30.0, (n, 1))
    return rng.normal(-5.0, 0.7, (n, 1)), p / MASS


def _ring_initial(case, seed):
    """Bead positions and velocities (ntraj, P) of thermal ring polymers in the left well, built from the
    normal modes of the free ring polymer with the well's frequency added."""
    rng, n, P = _rng(case, seed), case["ntraj"], case["beads"]
    wn, beta_p, w0 = P / RP_BETA, RP_BETA / P, math.sqrt(0.1 / RP_MASS)
    k, j = np.arange(P), np.arange(P)
    wk = 2 * wn * np.sin(np.pi * k / P)
    sd = 1.0 / np.sqrt(beta_p * RP_MASS * (wk ** 2 + w0 ** 2))
    sd[0] = min(sd[0], 0.5)   # a packet inside the well
    ang = 2 * np.pi * np.outer(j, k) / P
    basis = (np.cos(ang) + np.sin(ang)) / math.sqrt(P)
    modes = rng.standard_normal((n, P)) * sd
    r = modes @ basis.T - 3.87
    v = rng.standard_normal((n, P)) / math.sqrt(beta_p * RP_MASS) * 0.2
    return r, v


def _diatom_initial(case, seed):
    rng, n = _rng(case, seed), case["ntraj"]
    u = rng.standard_normal((n, 3))
    u /= np.linalg.norm(u, axis=1, keepdims=True)
    b = 2.2 + 0.1 * rng.standard_normal((n, 1))
    c = np.concatenate([rng.standard_normal((n, 2)), np.full((n, 1), 6.0)], axis=1)
    r0 = np.concatenate([c + 0.5 * b * u, c - 0.5 * b * u], axis=1)
    v0 = 2e-4 * rng.standard_normal((n, 6))
    v0[:, 2] -= 3e-3
    v0[:, 5] -= 3e-3
    return r0, v0


def _diatom_configurations(n, rng):
    u = rng.standard_normal((n, 3))
    u /= np.linalg.norm(u, axis=1, keepdims=True)
    b = 2.25 + 0.15 * rng.standard_normal((n, 1))
    c = np.concatenate([rng.standard_normal((n, 2)), rng.uniform(2.2, 9.0, (n, 1))], axis=1)
    return np.concatenate([c + 0.5 * b * u, c - 0.5 * b * u], axis=1)


@functools.lru_cache(maxsize=1)
def _surrogate_weights():
    """Two ensemble members for the diatom-surface model: random hidden layers, the last one fitted to the
    analytic model by least squares.  A few millihartree off, and the members seldom far apart."""
    X = _diatom_configurations(20000, np.random.default_rng(5))
    Y = NQ.DiatomSurface().potential(X)
    d = X[:, :3] - X[:, 3:]
    b = np.linalg.norm(d, axis=1)
    q = np.stack([b, X[:, 2], X[:, 5], d[:, 2] / b, 0.5 * (X[:, 0] + X[:, 3]), 0.5 * (X[:, 1] + X[:, 4])], axis=1)
    shift, scale, oshift, oscale = q.mean(0), 1.0 / q.std(0), Y.mean(0), Y.std(0)
    xn, tn = (q - shift) * scale, (Y - oshift) / oscale
    members = []
    for k in range(2):
        r = np.random.default_rng(100 + k)
        W1, b1 = r.normal(0, 0.5, (128, 6)), r.normal(0, 1.0, 128)
        W1[:, 4:] = 0.0
        W2, b2 = r.normal(0, 1 / math.sqrt(128), (128, 128)), r.normal(0, 0.3, 128)
        h = np.concatenate([np.tanh(np.tanh(xn @ W1.T + b1) @ W2.T + b2), np.ones((len(xn), 1))], axis=1)
        w = np.linalg.solve(h.T @ h + 1e-3 * np.eye(129), h.T @ tn)
        members.append(np.concatenate([a.reshape(-1) for a in (W1, b1, W2, b2, w[:128].T, w[128])]).astype(np.float32))
    return members, np.concatenate([shift, scale, oshift, oscale]).astype(np.float32)


def _pure(n, nstates):
    sig = np.zeros((n, nstates, nstates), complex)
    sig[:, 0, 0] = 1.0
    return sig


def _key(seed):
    return (0x4E5143444D493335 + 0x9E3779B97F4A7C15 * (int(seed) + 1)) & 0xFFFFFFFFFFFFFFFF


def _bath():
    w, c = NQ.DebyeSpectralDensity(5.0, 0.625).discretise(100)
    t = np.tanh(5.0 * w / 2)
    return w, c, np.sqrt(1 / (2 * w * t)), np.sqrt(w / (2 * t))


def prepare(case, seed):
    path, key = case["path"], _key(seed)
    if path == "call":
        method = {"fssh": NQ.FSSH, "ehrenfest": NQ.Ehrenfest}[case["method"]]
        sim = NQ.Simulation[method](NQ.Atoms(MASS), TULLY_MODEL[case["model"]]())
        p = 20.0
        dist = NQ.DynamicalDistribution(p / MASS, NQ.Normal(-5.0, p / (20 * math.sqrt(2))), (1, 1)) \
            * NQ.PureState(1, NQ.Adiabatic())
        return {"case": case, "sim": sim, "dist": dist, "ens": NQ.EnsembleMI355X(seed=key)}
    E = L.Ensemble(0)
    s = {"case": case, "E": E, "key": key}
    prec = L.PREC_FP32_NUCLEI if case.get("precision") == "fp32" else L.PREC_FP64
    if path == "mixed":
        E.set_problem(L.METHOD_FSSH, 2, 1, 1, [MASS], 1.0, precision=prec)
        for slot, k in enumerate((1, 2, 3)):
            E.set_model(slot, k - 1, TULLY[k])
        E.sample_initial(L.SAMPLER_TULLY_GRID, case["ntraj"], [-5.0, 5.0, 31], key, n_models=3)
    elif path == "two_state":
        E.set_problem(L.METHOD_FSSH if case["method"] == "fssh" else L.METHOD_EHRENFEST, 2, 1, 1, [MASS], 1.0)
        E.set_model(0, case["model"] - 1, TULLY[case["model"]])
        r, v = _two_state_initial(case, seed)
        E.load_initial(r, v, _pure(len(r), 2), state=np.zeros(len(r), np.int32))
    elif path == "spin_boson":
        w, c, sr, sv = _bath()
        E.set_problem(L.METHOD_FSSH if case["method"] == "fssh" else L.METHOD_EHRENFEST, 2, 1, 100, np.ones(100), 0.002,
                      precision=L.PREC_FP32_NUCLEI)
        E.set_model(0, L.MODEL_SPIN_BOSON, np.concatenate([[1.0, 1.0], w, c]))
        z = np.zeros(100)
        E.sample_initial(L.SAMPLER_HARMONIC_WIGNER, case["ntraj"], np.concatenate([z, sr, z, sv]), key, initial_state=0,
                         state_basis=1)
    elif path in ("rpmd", "rpsh"):
        hop = path == "rpsh"
        E.set_problem(L.METHOD_RPSH if hop else L.METHOD_RPMD, 2 if hop else 1, 1, 1, [RP_MASS], 1.0,
                      algorithm=L.ALG_BCB_TSIT5 if hop else L.ALG_BCB, nbeads=case["beads"],
                      precision=L.PREC_FP32_NUCLEI, temperature=1.0 / RP_BETA)
        E.set_model(0, L.MODEL_DW_GAUSSIAN, WELL if hop else [WELL[0], WELL[1], 0.0, 0.0, 1.0])
        r, v = _ring_initial(case, seed)
        E.load_initial(r, v, _pure(len(r), 2), state=np.zeros(len(r), np.int32) if hop else None)
    elif path == "diatom":
        model = NQ.DiatomSurface()
        E.set_problem(L.METHOD_FSSH, 2, 3, 2, DIATOM_MASS, 2.0, precision=L.PREC_FP32_NUCLEI)
        if case["surrogate"]:
            members, norm = _surrogate_weights()
            model = NQ.MLPSurrogate(model, members, norm, 0.03)
            E.set_model(0, model.kind, model.params())
            for k, p in enumerate(members):
                E.surrogate_set_params(k, p, norm)
        else:
            E.set_model(0, model.kind, model.params())
        r, v = _diatom_initial(case, seed)
        E.load_initial(r, v, _pure(len(r), 2), state=np.zeros(len(r), np.int32))
    elif path == "train":
        s["X"] = _diatom_configurations(case["samples"], _rng(case, seed))
        s["Y"] = NQ.DiatomSurface().potential(s["X"])
    elif path == "iesh":
        M, W = case["levels"], 3 * IESH_GAMMA
        E.set_problem(L.METHOD_IESH if case["method"] == "iesh" else L.METHOD_EHRENFEST_NA, M + 1, 1, 1, [MASS], 2.0,
                      algorithm=L.ALG_VERLET_ELECTRONICS, n_electrons=M // 2)
        E.set_model(0, L.MODEL_NEWNS_ANDERSON, [2000.0, 2e-4, 20.6097, -3.8e-3, IESH_GAMMA, -W, W, M])
        E.sample_initial(L.SAMPLER_GAUSSIAN, case["ntraj"], [8.0, 1.0, 0.0, 1e-2], key)
    elif path == "morse":
        rng, n = _rng(case, seed), case["ntraj"]
        E.set_problem(L.METHOD_FSSH, 3, 1, 1, [20000.0], 1.0, precision=prec)
        E.set_model(0, L.MODEL_MORSE_N, [3] + MORSE3_FSSH)
        r = rng.normal(3.0, 0.15, (n, 1))
        v = np.sqrt(2 * rng.uniform(0.02, 0.04, (n, 1)) / 20000.0)
        E.load_initial(r, v, _pure(n, 3), state=np.zeros(n, np.int32))
    else:
        n = case["nstates"]
        mass, gauss, dt = (2000.0, [-6.0, 0.5, 15.0 / 2000, 1.0 / 2000], 1.0) if n == 2 else \
            (20000.0, [4.1, 0.1, 0.0, 2e-4], 2.0)
        E.set_problem(L.METHOD_SPIN_MAPPING if case["method"] == "spin" else L.METHOD_ECMM, n, 1, 1, [mass], dt,
                      algorithm=L.ALG_MINT, mapping_gamma=0.0 if case["method"] == "spin" else 0.5)
        E.set_model(0, *((L.MODEL_TULLY1, TULLY[1]) if n == 2 else (L.MODEL_MORSE_N, [3] + MORSE3_MAP)))
        E.sample_initial(L.SAMPLER_GAUSSIAN, case["ntraj"], gauss, key, initial_state=0, state_basis=1)
    return s


# --- one pass ---------------------------------------------------------------------------------------
def run(state):
    case, path = state["case"], state["case"]["path"]
    if path == "call":
        sim, steps = state["sim"], case["nsteps"]
        out = (NQ.OutputAdiabaticPopulation, NQ.OutputDiabaticPopulation, NQ.OutputStateResolvedScattering1D(sim))
        every = np.arange(0, steps + 1, case["save_every"], dtype=np.float64)
        res = NQ.run_dynamics(sim, (0.0, float(steps)), state["dist"], output=out, reduction=NQ.MeanReduction(),
                              trajectories=case["ntraj"], dt=1.0, saveat=every, ensemble_algorithm=state["ens"])
        sc = res["OutputStateResolvedScattering1D"]
        return {"adiabatic": np.stack(res["OutputAdiabaticPopulation"]),
                "diabatic": np.stack(res["OutputDiabaticPopulation"]), "reflection": sc["reflection"],
                "transmission": sc["transmission"]}
    E, key = state["E"], state["key"]
    if path == "mixed":
        E.run(0.0, 10000.0, key, term=(0, 10.0))
        return {"population": E.reduce(L.OUT_FINAL_ADIABATIC_POPULATION, L.RED_MEAN, 2),
                "scattering": E.reduce(L.OUT_SCATTERING_1D, L.RED_MEAN, 4), "state": E.download(L.FIELD_STATE),
                "nhops": E.download(L.FIELD_NHOPS)}
    if path == "two_state":
        E.run(0.0, float(case["nsteps"]), key, save_every=case["save_every"])
        n = E.nsave
        return {"adiabatic": E.reduce(L.OUT_ADIABATIC_POPULATION, L.RED_MEAN, 2 * n),
                "diabatic": E.reduce(L.OUT_DIABATIC_POPULATION, L.RED_MEAN, 2 * n),
                "kinetic": E.reduce(L.OUT_KINETIC_ENERGY, L.RED_MEAN, n), "r": E.download(L.FIELD_R),
                "v": E.download(L.FIELD_V), "rho_re": E.download(L.FIELD_SIGMA_RE),
                "rho_im": E.download(L.FIELD_SIGMA_IM), "state": E.download(L.FIELD_STATE)}
    if path == "spin_boson":
        E.run(0.0, 0.002 * case["nsteps"], key, save_every=50)
        return {"correlation": E.reduce(L.OUT_POPULATION_CORRELATION, L.RED_MEAN, 4 * E.nsave),
                "diabatic": E.reduce(L.OUT_DIABATIC_POPULATION, L.RED_MEAN, 2 * E.nsave)}
    if path == "rpmd":
        E.run(0.0, float(case["nsteps"]), key, save_every=100)
        return {"centroid": E.reduce(L.OUT_CENTROID_POSITION, L.RED_MEAN, E.nsave), "r": E.download(L.FIELD_R)}
    if path == "rpsh":
        E.run(0.0, float(case["nsteps"]), key, save_every=100)
        return {"centroid": E.reduce(L.OUT_CENTROID_POSITION, L.RED_MEAN, E.nsave),
                "adiabatic": E.reduce(L.OUT_ADIABATIC_POPULATION, L.RED_MEAN, 2 * E.nsave),
                "state": E.download(L.FIELD_STATE), "nhops": E.download(L.FIELD_NHOPS)}
    if path == "diatom":
        E.run(0.0, 2.0 * case["nsteps"], key, save_every=100, term=(2, 8.0))
        return {"final": E.reduce(L.OUT_FINAL_ADIABATIC_POPULATION, L.RED_MEAN, 2),
                "adiabatic": E.reduce(L.OUT_ADIABATIC_POPULATION, L.RED_MEAN, 2 * E.nsave)}
    if path == "train":
        hist = E.surrogate_train(state["X"], state["Y"], steps=case["steps"], batch=case["batch"], lr=3e-3, lr_final=1e-4,
                                 seed=key)
        return {"loss": hist, "weights": np.stack([E.surrogate_get_params(k)[0] for k in range(2)])}
    if path == "iesh":
        E.run(0.0, 2.0 * case["nsteps"], key, save_every=10)
        n = case["levels"] + 1
        return {"adiabatic": E.reduce(L.OUT_ADIABATIC_POPULATION, L.RED_MEAN, n * E.nsave),
                "diabatic": E.reduce(L.OUT_DIABATIC_POPULATION, L.RED_MEAN, n * E.nsave), "r": E.download(L.FIELD_R),
                "v": E.download(L.FIELD_V), "nhops": E.download(L.FIELD_NHOPS)}
    if path == "morse":
        E.run(0.0, float(case["nsteps"]), key, save_every=100)
        return {"adiabatic": E.reduce(L.OUT_ADIABATIC_POPULATION, L.RED_MEAN, 3 * E.nsave),
                "diabatic": E.reduce(L.OUT_DIABATIC_POPULATION, L.RED_MEAN, 3 * E.nsave),
                "state": E.download(L.FIELD_STATE), "nhops": E.download(L.FIELD_NHOPS)}
    n = case["nstates"]
    E.run(0.0, (1.0 if n == 2 else 2.0) * case["nsteps"], key, save_every=100)
    return {"diabatic": E.reduce(L.OUT_DIABATIC_POPULATION, L.RED_MEAN, n * E.nsave),
            "correlation": E.reduce(L.OUT_POPULATION_CORRELATION, L.RED_MEAN, n * n * E.nsave),
            "energy": E.reduce(L.OUT_TOTAL_ENERGY, L.RED_MEAN, E.nsave), "x": E.download(L.FIELD_MAP_X)}


def work(case):
    """Initial conditions read and results written once; the arithmetic of one step of one trajectory: the
    model, its eigenstates and the coupling, a rotation of the density, and the nuclear step."""
    path, n = case["path"], case.get("ntraj", 1)
    if path in ("call", "two_state"):
        saves = case["nsteps"] // case["save_every"] + 1
        return {"bytes": n * (2 * 48 + 12 + 36 * saves), "flops": 300 * n * case["nsteps"]}
    if path == "mixed":
        return {"bytes": n * 120, "flops": 300 * 1750 * n}   # 1750 steps on average
    if path == "spin_boson":
        return {"bytes": n * (4 * 800 + 44 + 36 * (case["nsteps"] // 50 + 1)), "flops": (1200 + 250) * n * case["nsteps"]}
    if path in ("rpmd", "rpsh"):
        P = case["beads"]
        per = P * (4 * math.log2(P) + 20) + (P * 15 + 250 if path == "rpsh" else 0)
        saves = case["nsteps"] // 100 + 1
        return {"bytes": n * (32 * P + (8 + (36 if path == "rpsh" else 0)) * saves), "flops": per * n * case["nsteps"]}
    if path == "diatom":
        saves = case["nsteps"] // 100 + 1
        per = 2 * (4 * 2 * 128 * 128 + 4 * 2 * 6 * 128) + 400 if case["surrogate"] else 400
        return {"bytes": n * (4 * 48 + 80 + 36 * saves), "flops": per * n * case["nsteps"]}
    if path == "train":
        return {"bytes": 72 * case["samples"], "flops": 2 * 6 * (128 * 128 + 128 * 9) * case["steps"] * case["batch"]}
    if path == "iesh":
        N, ne = case["levels"] + 1, case["levels"] // 2
        saves = case["nsteps"] // 10 + 1
        return {"bytes": n * (32 * N * ne + 16 * N * saves), "flops": (8 * 4 * N * N * ne + 16 * N * N) * n * case["nsteps"]}
    saves = case["nsteps"] // 100 + 1
    if path == "morse":
        return {"bytes": n * (2 * 160 + 52 * saves), "flops": 1200 * n * case["nsteps"]}
    k = case["nstates"]
    return {"bytes": n * (32 + 32 * k + (8 * k + 16) * saves), "flops": (300 if k == 2 else 900) * n * case["nsteps"]}


def tolerance(case):
    """FP64 paths agree with 64-bit torch to about 1e-11 over these lengths.  FP32 beads: about 1e-6.  The other
    FP32 and BF16 paths: a hop decided the other way moves whole numbers of that trajectory, and means by a few
    parts in the number of trajectories; where rounding decorrelates trajectories, by their sampling error."""
    path = case["path"]
    n = case.get("ntraj", 1)
    if path in ("call", "two_state", "iesh", "mapping") or (path in ("mixed", "morse") and case["precision"] == "fp64"):
        return {"rel": 1e-8, "max": 1e-5, "differ": 1e-4}
    if path == "rpmd":
        return {"rel": 1e-5, "max": 1e-3}
    if path == "spin_boson":
        return {"rel": min(0.03, 2e-3 + 1.0 / math.sqrt(n)), "max": 0.2}
    if path == "train":
        return {"rel": 0.03, "max": 0.99}
    if path == "diatom":
        return {"rel": min(0.03, 1.0 / math.sqrt(n)), "max": 0.2}
    return {"rel": min(0.03, 2e-3 + 2.0 / n), "max": 0.1, "differ": 5e-3}


# --- the same in 64 bits, in torch ---------------------------------------------------------------------
_C = (0.161, 0.327, 0.9, 0.9800255409045097, 1.0)
_A = ((0.161,), (-0.008480655492356989, 0.335480655492357), (2.897153057105493, -6.359448489975075, 4.3622954328695815),
      (5.325864828439257, -11.748883564062828, 7.4955393428898365, -0.09249506636175525),
      (5.86145544294642, -12.92096931784711, 8.159367898576159, -0.071584973281401, -0.028269050394068383))
_B = (0.09646076681806523, 0.01, 0.4798896504144996, 1.379008574103742, -3.290069515436081, 2.324710524099774)
_M32 = 0xFFFFFFFF


def _philox(c0, c1, c2, c3, key):
    """Philox4x32-10 on int64 tensors that hold 32-bit values."""
    k0, k1 = key & _M32, key >> 32

    def mul(m, c):   # high and low words of a 32 x 32 bit product, from 16-bit halves
        lo, hi = m * (c & 0xFFFF), m * (c >> 16)
        t = hi + (lo >> 16)
        return (t >> 16) & _M32, ((t & 0xFFFF) << 16) | (lo & 0xFFFF)
    for _ in range(10):
        h0, l0 = mul(0xD2511F53, c0)
        h1, l1 = mul(0xCD9E8D57, c2)
        c0, c1, c2, c3 = h1 ^ c1 ^ k0, l1, h0 ^ c3 ^ k1, l0
        k0, k1 = (k0 + 0x9E3779B9) & _M32, (k1 + 0xBB67AE85) & _M32
    return c0, c1, c2, c3


def _u53(a, b):
    return (((a << 21) | (b >> 11)).double()) * 2.0 ** -53


def _uniform(tid, step, stream, key):
    z = torch.zeros_like(tid)
    c0, c1, _, _ = _philox(tid, z, z + step, z + stream, key)
    return _u53(c0, c1)


def _normal2(tid, dof, key):
    z = torch.zeros_like(tid)
    c = _philox(tid, z, z + dof, z, key)
    rad = torch.sqrt(-2.0 * torch.log(1.0 - _u53(c[0], c[1])))
    u = 2 * math.pi * _u53(c[2], c[3])
    return rad * torch.cos(u), rad * torch.sin(u)


def _tully(model, x):
    p = TULLY[model]
    if model == 1:
        e, w = torch.exp(-p[1] * x.abs()), p[2] * torch.exp(-p[3] * x * x)
        v, d = p[0] * (1 - e) * torch.sign(x), p[0] * p[1] * e
        return v, -v, w, d, -d, -2 * p[3] * x * w
    if model == 2:
        g, w = p[0] * torch.exp(-p[1] * x * x), p[2] * torch.exp(-p[3] * x * x)
        z = torch.zeros_like(x)
        return z, p[4] - g, w, z, 2 * p[1] * x * g, -2 * p[3] * x * w
    e = torch.exp(-p[2] * x.abs())
    o = torch.ones_like(x)
    return p[0] * o, -p[0] * o, torch.where(x < 0, p[1] * e, p[1] * (2 - e)), 0 * o, 0 * o, p[1] * p[2] * e


def _eigen(a, c, d, prev):
    h = 0.5 * (a - d)
    rad = torch.sqrt(h * h + c * c)
    m = 0.5 * (a + d)
    up = h >= 0
    p, q = torch.where(up, h + rad, c), torch.where(up, c, rad - h)
    n = torch.sqrt(p * p + q * q)
    p, q = p / n, q / n
    lo, hi = (-q, p), (p, q)   # columns
    if prev is None:
        f0 = torch.where(torch.where(lo[1].abs() > lo[0].abs(), lo[1], lo[0]) < 0, -1.0, 1.0)
        f1 = torch.where(torch.where(hi[1].abs() > hi[0].abs(), hi[1], hi[0]) < 0, -1.0, 1.0)
    else:
        f0 = torch.where(lo[0] * prev[0] + lo[1] * prev[2] < 0, -1.0, 1.0)
        f1 = torch.where(hi[0] * prev[1] + hi[1] * prev[3] < 0, -1.0, 1.0)
    return m - rad, m + rad, (f0 * lo[0], f1 * hi[0], f0 * lo[1], f1 * hi[1])


def _two_state_exact(hop, model, r, v, nsteps, save_every, key):
    """B-A-B velocity Verlet with five Tsit5 sub-steps of the density and the hop after each step."""
    tid = torch.arange(len(r), device=r.device)
    q, x, y = torch.ones_like(r), torch.zeros_like(r), torch.zeros_like(r)
    st = torch.zeros_like(tid)

    def cache(prev):
        a, d, c, da, dd, dc = _tully(model, r)
        E0, E1, U = _eigen(a, c, d, prev)
        g = lambda i, j: U[i] * U[j] * da + (U[i] * U[j + 2] + U[i + 2] * U[j]) * dc + U[i + 2] * U[j + 2] * dd  # noqa: E731
        return E0, E1, U, g(0, 0), g(1, 1), g(0, 1)

    def accel(G0, G1, G01):
        f = torch.where(st == 0, G0, G1) if hop else G0 * 0.5 * (1 + q) + G1 * 0.5 * (1 - q) + 2 * G01 * x
        return -f / MASS
    E0, E1, U, G0, G1, G01 = cache(None)
    k = accel(G0, G1, G01)
    dEc, wc, ad, di, ek = 0 * r, 0 * r, [], [], []

    def save():
        pa = torch.where(st == 0, 1.0, 0.0).double() if hop else 0.5 * (1 + q)
        pb = 1 - pa
        ad.extend([pa.mean(), pb.mean()])
        di.extend([(U[i] ** 2 * pa + U[i + 1] ** 2 * pb + 2 * U[i] * U[i + 1] * x).mean() for i in (0, 2)])
        ek.append((0.5 * MASS * v * v).mean())
    save()
    h = 0.2
    for step in range(nsteps):
        vt = v + 0.5 * k
        r = r + vt
        E0, E1, U, G0, G1, G01 = cache(U)
        k = accel(G0, G1, G01)
        v = vt + 0.5 * k
        d01 = G01 / (E1 - E0)
        w, dE = d01 * v, E0 - E1
        sE, sw = dE - dEc, w - wc
        for s in range(5):
            K = []
            for i in range(6):
                loc = h * (s + (0.0 if i == 0 else _C[i - 1]))
                e, g = dEc + sE * loc, 2 * (wc + sw * loc)
                u = [q, x, y]
                if i:
                    u = [b + h * sum(a * kk[m] for a, kk in zip(_A[i - 1], K)) for m, b in enumerate(u)]
                K.append((-2 * g * u[1], e * u[2] + 0.5 * g * u[0], -e * u[1]))
            q, x, y = (b + h * sum(a * kk[m] for a, kk in zip(_B, K)) for m, b in enumerate((q, x, y)))
        dEc, wc = dE, w
        if (step + 1) % save_every == 0:
            save()
        if hop:
            sgn = torch.where(st == 0, 1.0, -1.0).double()
            prob = 2 * v * (x / (0.5 * (1 + sgn * q))) * sgn * d01
            want = prob.clamp(0, 1) > _uniform(tid, step, 1, key)
            dm, gap = -sgn * d01, sgn * (E1 - E0)
            a, b = 0.5 * dm * dm / MASS, dm * v
            disc = b * b - 4 * a * gap
            want &= disc >= 0
            root = torch.sqrt(disc.clamp(min=0))
            gam = torch.where(b < 0, b + root, b - root) / (2 * a)
            v = torch.where(want, v - gam * dm / MASS, v)
            st = torch.where(want, 1 - st, st)
    cat = lambda z: torch.stack(z).cpu().numpy()  # noqa: E731
    return {"adiabatic": cat(ad), "diabatic": cat(di), "kinetic": cat(ek), "r": r, "v": v, "q": q, "x": x, "y": y, "st": st}


def _ring_exact(case, seed, dev):
    r, v = (torch.from_numpy(a).to(dev) for a in _ring_initial(case, seed))
    P = case["beads"]
    wn = P / RP_BETA
    j = torch.arange(P, device=dev, dtype=torch.float64)
    ang = 2 * math.pi * torch.outer(j, j) / P
    H = (torch.cos(ang) + torch.sin(ang)) / math.sqrt(P)
    wk = 2 * wn * torch.sin(math.pi * j / P)
    den = 1 + wk ** 2 / 4
    c11, c12, c21 = (1 - wk ** 2 / 4) / den, 1 / den, -wk ** 2 / den
    force = lambda x: -(4 * WELL[0] * x ** 3 - 2 * WELL[1] * x)  # noqa: E731
    f, out = force(r), [r.mean()]
    for step in range(case["nsteps"]):
        v = v + 0.5 * f / RP_MASS
        q, p = r @ H, v @ H
        r, v = (c11 * q + c12 * p) @ H, (c21 * q + c11 * p) @ H
        f = force(r)
        v = v + 0.5 * f / RP_MASS
        if (step + 1) % 100 == 0:
            out.append(r.mean())
    return {"centroid": torch.stack(out).cpu().numpy(), "r": r.cpu().numpy()}


def exact(case, seed):
    """None for the paths whose trajectories part ways at rounding level (hops in FP32, a stiff bath, BF16
    weights), and for those that need an eigen-decomposition a step and so over 20 seconds."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    path = case["path"]
    if path == "rpmd":
        return _ring_exact(case, seed, dev)
    if path not in ("call", "two_state"):
        return None
    n, hop, key = case["ntraj"], case["method"] == "fssh", _key(seed)
    if path == "call":
        z0, _ = _normal2(torch.arange(n, device=dev), 0, key)
        r = -5.0 + 20.0 / (20 * math.sqrt(2)) * z0
        e = _two_state_exact(hop, case["model"], r, torch.full_like(r, 20.0 / MASS), case["nsteps"], case["save_every"], key)
        pops = torch.stack([1.0 - e["st"].double(), e["st"].double()], 1) if hop else \
            torch.stack([0.5 * (1 + e["q"]), 0.5 * (1 - e["q"])], 1)
        right = (e["r"] > 0).double()[:, None]
        return {"adiabatic": e["adiabatic"].reshape(-1, 2), "diabatic": e["diabatic"].reshape(-1, 2),
                "reflection": (pops * (1 - right)).mean(0).cpu().numpy(), "transmission": (pops * right).mean(0).cpu().numpy()}
    r, v = (torch.from_numpy(a[:, 0].copy()).to(dev) for a in _two_state_initial(case, seed))
    e = _two_state_exact(hop, case["model"], r, v, case["nsteps"], case["save_every"], key)
    a, b, z = 0.5 * (1 + e["q"]), 0.5 * (1 - e["q"]), torch.zeros_like(e["q"])
    mat = lambda *m: torch.stack(m, 1).reshape(-1, 2, 2).cpu().numpy()  # noqa: E731
    return {"adiabatic": e["adiabatic"], "diabatic": e["diabatic"], "kinetic": e["kinetic"],
            "r": e["r"][:, None].cpu().numpy(), "v": e["v"][:, None].cpu().numpy(),
            "rho_re": mat(a, e["x"], e["x"], b), "rho_im": mat(z, e["y"], -e["y"], z), "state": None}
