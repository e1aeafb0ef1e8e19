"""Performance cases: what programs have this library do, through its
public entry points, over the range of system sizes, active sets,
precisions and batch shapes it is used with.

Kinds (case["kind"]):

update    one h4h_update_acc_jrk_static call on device arrays (C ABI), the
          smallest unit of work: a caller that drives its own integrator.
forces    Hermite4HIP.init_acc_jrk: the forces of all n particles, and their
          download.
energy    Hermite4HIP.get_energy: the O(n^2) energy of an output time.
run       an integration from initial conditions on a context in hand:
          upload, initial forces, steps and energy, the first max_steps block
          steps on the device, the energy there, and the state's download
          (what a snapshot needs).
steps     the same driven from the host, one h4h_step call per block step.
ensemble  a batch of independent clusters on a handle in hand: upload, the
          whole integration to t_end with its energies, download.

Initial conditions are seeded Plummer spheres in Henon units, eps = 1e-4,
eta = 0.01, as in this repository's benchmark and tests.
"""
import ctypes
import math

import numpy as np
import torch

import gravidy_amd
from gravidy_amd import EnsembleHIP, Hermite4HIP, ic, softening_e2

EPS = 1e-4
STATE = ("r", "v", "f", "t", "dt")  # what a snapshot or a restart holds
FLOPS_PAIR = 60        # one Hermite pair interaction, by convention
FLOPS_ENERGY_PAIR = 16  # 3 sub, 3 FMA, 1/r with one refinement, 1 FMA
PRECISION = {"fp64": gravidy_amd.H4H_FP64, "exact": gravidy_amd.H4H_FP64_EXACT,
             "mixed": gravidy_amd.H4H_MIXED}


def listed():
    return [
        # A caller's own integrator loop: a handful of active particles of a
        # small system, one call per block step; latency is everything.
        {"name": "update_n1024_act24", "kind": "update", "n": 1024, "nact": 24,
         "precision": "fp64"},
        # A host-driven loop (one library call per block step), as a program
        # that inspects every step runs it.
        {"name": "steps_n4096", "kind": "steps", "n": 4096, "max_steps": 256,
         "precision": "fp64"},
        # The flagship kernel: the initial forces of the headline workload.
        {"name": "forces_n262144", "kind": "forces", "n": 262144, "precision": "fp64"},
        # The same in mixed precision at a ragged size.
        {"name": "forces_mixed_n100003", "kind": "forces", "n": 100003, "precision": "mixed"},
        # Energy check of a production snapshot.
        {"name": "energy_n131072", "kind": "energy", "n": 131072},
        # The smallest configuration as users run it, about to its first output.
        {"name": "run_n1024", "kind": "run", "n": 1024, "max_steps": 800, "precision": "fp64"},
        # An open-cluster size, ragged: block steps with small active sets.
        {"name": "run_n10007", "kind": "run", "n": 10007, "max_steps": 640,
         "precision": "fp64"},
        # The single-GPU configuration's first stretch.
        {"name": "run_n65536", "kind": "run", "n": 65536, "max_steps": 512,
         "precision": "fp64"},
        # The mixed-precision configuration's first stretch.
        {"name": "run_mixed_n262144", "kind": "run", "n": 262144, "max_steps": 128,
         "precision": "mixed"},
        # A bit-exact reference run (regression of a published run).
        {"name": "run_exact_n1024", "kind": "run", "n": 1024, "max_steps": 64,
         "precision": "exact"},
        # The ensemble configuration: 64 clusters of 1024 to 32768 stars.
        {"name": "ensemble_64_uneven", "kind": "ensemble", "clusters": 64, "nmin": 1024,
         "nmax": 32768, "sizes_seed": 64, "t_end": 0.00390625, "precision": "fp64"},
        # A parameter study: many small clusters.
        {"name": "ensemble_256_small", "kind": "ensemble", "clusters": 256, "nmin": 128,
         "nmax": 1024, "sizes_seed": 256, "t_end": 0.0625, "precision": "fp64"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["update", "forces", "energy", "run", "run", "run", "steps", "ensemble"])
    if kind == "update":
        n = _log_int(rng, 64, 65536)
        return {"kind": kind, "n": n, "nact": _log_int(rng, 1, n),
                "precision": rng.choice(["fp64", "fp64", "mixed"])}
    if kind == "forces":
        precision = rng.choice(["fp64", "fp64", "mixed", "exact"])
        return {"kind": kind, "n": _log_int(rng, 100, 16384 if precision == "exact" else 262144),
                "precision": precision}
    if kind == "energy":
        return {"kind": kind, "n": _log_int(rng, 100, 262144)}
    if kind == "steps":
        return {"kind": kind, "n": _log_int(rng, 64, 32768), "max_steps": rng.randint(16, 256),
                "precision": rng.choice(["fp64", "mixed"])}
    if kind == "ensemble":
        nmax = rng.choice([1024, 4096, 16384])
        return {"kind": kind, "clusters": rng.randint(8, 96), "nmin": nmax // 16, "nmax": nmax,
                "sizes_seed": rng.randint(1, 10 ** 6), "t_end": 2.0 ** -rng.randint(6, 8),
                "precision": rng.choice(["fp64", "mixed"])}
    precision = rng.choice(["fp64", "fp64", "mixed", "exact"])
    if precision == "exact":
        return {"kind": kind, "n": _log_int(rng, 64, 8192), "max_steps": rng.randint(4, 32),
                "precision": precision}
    return {"kind": kind, "n": _log_int(rng, 64, 131072), "max_steps": rng.randint(32, 512),
            "precision": precision}


def _sizes(case):
    return [int(k) for k in ic.log_uniform_sizes(case["clusters"], case["sizes_seed"],
                                                 case["nmin"], case["nmax"])]


def _active(n, nact, seed):
    return np.random.default_rng(seed).choice(n, nact, replace=False).astype(np.uint32)


def _check(lib, rc):
    if rc:
        raise RuntimeError(lib.h4h_last_error().decode())


def prepare(case, seed):
    e2 = softening_e2(EPS)
    if case["kind"] == "ensemble":
        systems = [ic.plummer(n, 1000 * seed + k) for k, n in enumerate(_sizes(case))]
        n = sum(r.shape[0] for r, _ in systems)
        return {"case": case, "ens": EnsembleHIP(systems, e2, precision=case["precision"]),
                "r": np.concatenate([r for r, _ in systems]),
                "v": np.concatenate([v for _, v in systems]),
                "state": {"r": np.zeros((n, 4)), "v": np.zeros((n, 4)), "f": np.zeros((n, 6)),
                          "t": np.zeros(n), "dt": np.zeros(n)}}
    n = case["n"]
    r, v = ic.plummer(n, seed)
    if case["kind"] == "update":
        dev = torch.device("cuda")
        p6 = np.concatenate([r[:, :3], v[:, :3]], axis=1)
        move = _active(n, case["nact"], seed)
        return {"case": case, "e2": e2, "lib": gravidy_amd.load(),
                "p6": torch.tensor(p6, device=dev),
                "pm": torch.tensor(r[:, 3].astype(np.float32), device=dev),
                "move": torch.tensor(move.astype(np.int32), device=dev),
                "f6": torch.zeros((n, 6), dtype=torch.float64, device=dev)}
    h = Hermite4HIP(r, v, e2, precision=case.get("precision", "fp64"))
    return {"case": case, "e2": e2, "r": r, "v": v, "h": h}


def _dp(a):
    return a.ctypes.data_as(ctypes.POINTER(ctypes.c_double))


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "update":
        _check(state["lib"], state["lib"].h4h_update_acc_jrk_static(
            state["p6"].data_ptr(), state["pm"].data_ptr(), case["n"], state["move"].data_ptr(),
            case["nact"], state["e2"], PRECISION[case["precision"]], state["f6"].data_ptr(),
            torch.cuda.current_stream().cuda_stream))
        return state["f6"]
    if kind == "forces":
        state["h"].init_acc_jrk()
        return state["h"].download()["f"]
    if kind == "energy":
        return state["h"].get_energy()
    if kind == "ensemble":
        ens = state["ens"]
        # The Python class uploads when it is made and downloads into one new
        # array per cluster; a program that keeps its handle and arrays calls
        # the ABI for both.
        _check(ens.lib, ens.lib.h4h_upload(ens._ctx, _dp(state["r"]), _dp(state["v"]), None, None,
                                           None))
        out = ens.integration(case["t_end"], interval=case["t_end"])
        _check(ens.lib, ens.lib.h4h_download(ens._ctx, *(_dp(state["state"][k]) for k in STATE),
                                             None, None, None))
        out.update(state["state"])
        return out
    h = state["h"]
    h.upload(state["r"], state["v"])
    if kind == "steps":
        out = h.integration(1.0, interval=1.0, max_steps=case["max_steps"], mode="step")
    else:
        out = h.integration(1.0, interval=1.0, max_steps=case["max_steps"])
        out["energy_end"] = h.get_energy()
    d = h.download()
    out.update({k: d[k] for k in STATE})
    return out


def work(case):
    kind = case["kind"]
    if kind == "ensemble":
        sizes = _sizes(case)
    else:
        n = case["n"]
    if kind == "update":
        k = case["nact"]
        return {"bytes": n * 52 + k * (4 + 48), "flops": FLOPS_PAIR * k * n}
    if kind == "forces":
        return {"bytes": n * (64 + 48), "flops": FLOPS_PAIR * n * n}
    if kind == "energy":
        return {"bytes": n * 64, "flops": FLOPS_ENERGY_PAIR * n * (n - 1) // 2}

    # Whole runs: the initial forces, two energies, and the block steps.  The
    # steps' pair interactions depend on the schedule: a block step of the
    # first hundreds moves about n / 128 particles on average, and to t_end a
    # particle makes 735 (n / 262144)^0.19 steps per unit time.
    def pairs(n):
        if kind == "ensemble":
            return n * n * case["t_end"] * 735.0 * (n / 262144.0) ** 0.19
        return case["max_steps"] * max(1.0, n / 128.0) * n

    sizes = sizes if kind == "ensemble" else [n]
    flops = sum(FLOPS_PAIR * (n * n + pairs(n)) + FLOPS_ENERGY_PAIR * n * n for n in sizes)
    # uploaded r, v; downloaded r, v, f, t, dt; a block step's own traffic is
    # the active particles' state, small beside the pairs
    return {"bytes": sum(n * (8 + 16) * 8 for n in sizes), "flops": flops}


def _exact_forces(r, v, m32, e2, active=None):
    """Accelerations and jerks by plain 64-bit sums over all pairs."""
    dev = torch.device("cuda")
    x, u, m = (torch.tensor(a, device=dev, dtype=torch.float64) for a in (r, v, m32))
    n = x.shape[0]
    rows = torch.arange(n, device=dev) if active is None else torch.tensor(
        active.astype(np.int64), device=dev)
    out = torch.empty((rows.numel(), 6), dtype=torch.float64, device=dev)
    step = max(1, (1 << 28) // n)
    for b in range(0, rows.numel(), step):
        i = rows[b:b + step]
        d = [x[None, :, k] - x[i, None, k] for k in range(3)]
        w = [u[None, :, k] - u[i, None, k] for k in range(3)]
        r2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2] + e2
        mr3 = m[None, :] / (r2 * torch.sqrt(r2))
        c = 3.0 * (d[0] * w[0] + d[1] * w[1] + d[2] * w[2]) / r2
        for k in range(3):
            out[b:b + step, k] = (mr3 * d[k]).sum(1)
            out[b:b + step, 3 + k] = (mr3 * (w[k] - c * d[k])).sum(1)
    return out.cpu().numpy()


def _exact_energy(r, v):
    dev = torch.device("cuda")
    x = torch.tensor(r[:, :3], device=dev)
    m = torch.tensor(r[:, 3], device=dev)
    n = x.shape[0]
    step = max(1, (1 << 28) // n)
    j = torch.arange(n, device=dev)
    pot = 0.0
    for b in range(0, n, step):
        d = torch.zeros((min(step, n - b), n), dtype=torch.float64, device=dev)
        for k in range(3):
            d += (x[None, :, k] - x[b:b + step, None, k]) ** 2
        t = m[b:b + step, None] * m[None, :] / torch.sqrt(d)
        t[j[None, :] <= j[b:b + step, None]] = 0.0
        pot -= float(t.sum())
    kin = float((0.5 * r[:, 3] * (v[:, :3] ** 2).sum(1)).sum())
    return kin, pot


def exact(case, seed):
    """Forces and energies by plain 64-bit sums.  A run's block steps have no
    closed value; its initial energy has."""
    kind = case["kind"]
    e2 = softening_e2(EPS)
    if kind == "ensemble":
        return None
    n = case["n"]
    r, v = ic.plummer(n, seed)
    m32 = r[:, 3].astype(np.float32).astype(np.float64)
    if kind == "forces":
        return _exact_forces(r[:, :3], v[:, :3], m32, e2)
    if kind == "update":
        move = _active(n, case["nact"], seed)
        f = np.zeros((n, 6))
        f[move] = _exact_forces(r[:, :3], v[:, :3], m32, e2, move)
        return f
    ek, ep = _exact_energy(r, v)
    if kind == "energy":
        return ek, ep
    if kind == "steps":
        return {"energy": np.array([ek + ep])}
    return {"energy_ini": ek + ep}
