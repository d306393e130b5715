"""The work a user of this package has it do, as cases that can be timed.

Every case goes through the package's public entry points (gpu.Sim,
gpu.Ensemble, surrogate.Net, the stateless stage calls and the C ABI's
device-buffer call).  The channels are the Poiseuille set of
params.poiseuille_params: 50x50 cells of 10 particles (the reference's
benchmark channel) up to 2048x1024 cells of 20, with the 1024x512x20 channel
of bench.py between them; ragged grids, low densities, moving and no-slip
walls and the threshold options are taken as well.

listed() gives the named cases, draw(rng) one more of the same ranges,
prepare(case, seed) the state a program holds before the call, run(state) one
pass, work(case) the bytes and operations a pass cannot do without, and
exact(case, seed) the results in 64 bits where plain torch or numpy can give
them (the stepping paths follow counter-based draws and have none).
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

from src_incompressible_openmp_amd import gpu, surrogate
from src_incompressible_openmp_amd.params import LAYOUT_BASE, LAYOUT_SHIFTED, poiseuille_params, to_struct

CHANNELS = (4, 32, 32, 32, 2)  # the surrogate network's layers
FIELDS = ("Ux", "Uy", "Px", "Py", "T", "rho", "Pkin", "Pvir", "P", "rhoTarget")
# compulsory particle traffic of one step (as bench.py counts it) and of one
# state download (x and v)
STEP_BYTES, STATE_BYTES = 256, 32


def listed():
    return [
        # one cell-field evaluation on device buffers, the call a serving or
        # monitoring loop makes on every frame: the smallest call, all launches
        {"name": "fields_50x50", "path": "fields", "Nx": 50, "Ny": 50, "ppc": 10},
        # the reference's benchmark channel: 100 steps between two dumps; a
        # handful of zones, so each step's chain of launches is what it takes
        {"name": "channel_50x50", "path": "channel", "Nx": 50, "Ny": 50, "ppc": 10, "steps": 100, "variant": "plain"},
        # an ordinary channel: fewer zones than the chip has CUs
        {"name": "channel_256x128", "path": "channel", "Nx": 256, "Ny": 128, "ppc": 20, "steps": 50,
         "variant": "plain"},
        # a ragged grid of low density with a moving and a no-slip wall, local
        # thresholds, mean flow removed, no zone or cell count even
        {"name": "channel_ragged_walls", "path": "channel", "Nx": 333, "Ny": 117, "ppc": 7, "steps": 50,
         "variant": "walls"},
        # the benchmark workload of bench.py
        {"name": "channel_1024x512", "path": "channel", "Nx": 1024, "Ny": 512, "ppc": 20, "steps": 100,
         "variant": "plain"},
        # a large instance: many more zones than fit the chip at once
        {"name": "channel_2048x1024", "path": "channel", "Nx": 2048, "Ny": 1024, "ppc": 20, "steps": 100,
         "variant": "plain"},
        # a run that writes its metrics row after every step, as the driver
        # with metricsEvery = 1 does
        {"name": "metrics_256x128", "path": "metrics", "Nx": 256, "Ny": 128, "ppc": 20, "steps": 20},
        # the benchmark workload with the closure surrogate on 49 of 50 steps
        {"name": "surrogate_1024x512", "path": "surrogate", "Nx": 1024, "Ny": 512, "ppc": 20, "steps": 50},
        # the network alone: evaluation of a stored snapshot, and the loss
        # and gradient of one mini-batch of its training
        {"name": "net_forward_1024x512", "path": "net_forward", "Nx": 1024, "Ny": 512, "batch": 1},
        {"name": "net_grad_256x128", "path": "net_grad", "Nx": 256, "Ny": 128, "batch": 4},
        # the stateless stage calls on host arrays, one step's worth: the
        # drop-in user's program, which keeps its state on the host
        {"name": "stages_256x128", "path": "stages", "Nx": 256, "Ny": 128, "ppc": 20},
        # a parameter study: uneven replicas stepped together
        {"name": "ensemble_24", "path": "ensemble", "replicas": 24, "layout": 2, "steps": 40},
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _grid(rng, cells_lo, cells_hi):
    cells, aspect = _log(rng, cells_lo, cells_hi), _log(rng, 1.0, 4.0)
    return max(32, int(round(math.sqrt(cells * aspect)))), max(24, int(round(math.sqrt(cells / aspect))))


def draw(rng):
    path = rng.choice(["channel"] * 6 + ["fields", "fields", "metrics", "surrogate", "net_forward", "net_grad", "stages",
                                         "ensemble"])
    if path == "channel":
        Nx, Ny = _grid(rng, 2500, 1.2e6)
        ppc = rng.randint(5, 24)
        steps = int(min(_log(rng, 20, 120), 2.5e9 / (Nx * Ny * ppc)))
        return {"path": path, "Nx": Nx, "Ny": Ny, "ppc": ppc, "steps": steps,
                "variant": rng.choice(["plain", "plain", "walls"])}
    if path == "fields":
        Nx, Ny = _grid(rng, 1500, 50000)
        return {"path": path, "Nx": Nx, "Ny": Ny, "ppc": rng.randint(5, 20)}
    if path == "metrics":
        Nx, Ny = _grid(rng, 2500, 2e5)
        return {"path": path, "Nx": Nx, "Ny": Ny, "ppc": rng.randint(5, 20), "steps": rng.randint(5, 25)}
    if path == "surrogate":
        Nx, Ny = _grid(rng, 2500, 6e5)
        return {"path": path, "Nx": Nx, "Ny": Ny, "ppc": rng.randint(8, 20), "steps": rng.randint(15, 60)}
    if path == "net_forward":
        Nx, Ny = _grid(rng, 2500, 6e5)
        return {"path": path, "Nx": Nx, "Ny": Ny, "batch": rng.randint(1, max(1, min(4, int(1e6 / (Nx * Ny)))))}
    if path == "net_grad":
        Nx, Ny = _grid(rng, 2500, 1e5)
        return {"path": path, "Nx": Nx, "Ny": Ny, "batch": rng.randint(1, 4)}
    if path == "stages":
        Nx, Ny = _grid(rng, 2500, 1e5)
        return {"path": path, "Nx": Nx, "Ny": Ny, "ppc": rng.randint(5, 20)}
    return {"path": path, "replicas": rng.randint(3, 28), "layout": rng.randint(1, 10 ** 6), "steps": rng.randint(10, 40)}


# ---- parameters ----

def _params(case):
    over = {}
    if case.get("variant") == "walls":
        over = dict(boundary_bottom="bounceback", Utop=0.3, useLocalFluidFractionThresholds=True, highMode="1+coef",
                    lowMode="1+coef", coef=0.2, lowThrFloor=0.5 * case["ppc"], highThrFloor=1.3 * case["ppc"],
                    keepMeanFlow=True, alpha=math.radians(130.0))
    return to_struct(poiseuille_params(Nx=case["Nx"], Ny=case["Ny"], gamma=float(case["ppc"]), **over))


def _replicas(case):
    """Uneven channels in the ranges of bench.py's ensemble."""
    rng = np.random.default_rng(case["layout"])
    ps = []
    for _ in range(case["replicas"]):
        nx, ny, ppc = int(rng.integers(64, 513)), int(rng.integers(32, 257)), int(rng.integers(5, 21))
        ps.append(to_struct(poiseuille_params(Nx=nx, Ny=ny, gamma=float(ppc),
                                              bodyForceX=float(10.0 ** rng.uniform(-4.0, -2.0)))))
    return ps


def _rho_target(p):
    return p.gamma / ((p.Lx / p.Nx) * (p.Ly / p.Ny))


# ---- inputs ----

def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _particles(p, gen):
    """Uniform positions and Maxwell velocities without mean, [n, 2] each."""
    x = torch.rand(p.n, 2, dtype=torch.float64, device="cuda", generator=gen)
    x *= torch.tensor([p.Lx, p.Ly], dtype=torch.float64, device="cuda")
    v = torch.randn(p.n, 2, dtype=torch.float64, device="cuda", generator=gen) * math.sqrt(p.kBT)
    v -= v.mean(dim=0)
    return x, v


def _host_particles(p, gen):
    return [a.cpu().numpy().reshape(-1) for a in _particles(p, gen)]


def _theta():
    """He-uniform weights and zero biases of the network."""
    rng = np.random.default_rng(1)
    parts = []
    for ci, co in zip(CHANNELS[:-1], CHANNELS[1:]):
        bound = math.sqrt(6.0 / (9 * ci))
        parts += [rng.uniform(-bound, bound, co * 9 * ci), np.zeros(co)]
    return np.concatenate(parts)


def _samples(case, seed):
    """Features and targets of closure snapshots: occupancy deviation, local
    velocity deviation and temperature deviation of cells of about 20
    particles, and a correction of unit scale."""
    gen = _generator(seed)
    shape = (case["batch"], case["Nx"] * case["Ny"])
    scale = torch.tensor([0.08, 0.25, 0.25, 0.23], device="cuda")
    f = torch.randn(*shape, 4, device="cuda", generator=gen) * scale
    t = torch.randn(*shape, 2, device="cuda", generator=gen)
    return f.cpu().numpy(), t.cpu().numpy()


def prepare(case, seed):
    path = case["path"]
    state = {"case": case}
    if path in ("net_forward", "net_grad"):
        net = surrogate.Net(case["Nx"], case["Ny"], True, False, max_batch=case["batch"])
        net.set_params(_theta())
        state["net"] = net
        state["features"], state["targets"] = _samples(case, seed)
        return state
    gen = _generator(seed)
    if path == "ensemble":
        ps = _replicas(case)
        ens = gpu.Ensemble(ps, [r + 1 for r in range(len(ps))])
        for r, p in enumerate(ps):
            ens.set_state(r, *_host_particles(p, gen))
        state.update(ens=ens, step=1)
        return state
    p = _params(case)
    state["p"] = p
    if path == "fields":
        x, v = _particles(p, gen)
        out = {"N": torch.zeros(p.Nc, dtype=torch.int32, device="cuda")}
        out.update({k: torch.zeros(p.Nc, dtype=torch.float64, device="cuda") for k in FIELDS})
        dp, ip = ctypes.POINTER(ctypes.c_double), ctypes.POINTER(ctypes.c_int32)
        state.update(x=x, v=v, out=out, lib=gpu.load(), rho=ctypes.c_double(_rho_target(p)),
                     xp=ctypes.cast(x.data_ptr(), dp), vp=ctypes.cast(v.data_ptr(), dp),
                     fields=gpu.CellFieldsC(ctypes.cast(out["N"].data_ptr(), ip),
                                            *[ctypes.cast(out[k].data_ptr(), dp) for k in FIELDS]))
        return state
    x, v = _host_particles(p, gen)
    if path == "stages":
        state.update(x=x, v=v, step=1)
        return state
    sim = gpu.Sim(p)
    sim.set_state(x, v)
    state.update(sim=sim, step=1)
    if path == "surrogate":
        net = surrogate.Net(p.Nx, p.Ny, True, False, max_batch=1)
        net.set_params(_theta())
        sim.set_surrogate(net, 50, 1e-3, 5e-2)
        state["net"] = net
    return state


# ---- one pass ----

def run(state):
    case = state["case"]
    path = case["path"]
    if path == "fields":
        gpu._check(state["lib"].mpcd_gpu_compute_cell_fields_noalloc(
            ctypes.byref(state["p"]), state["xp"], state["vp"], state["rho"], ctypes.byref(state["fields"]),
            ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
        return state["out"]
    if path == "net_forward":
        return state["net"].forward(state["features"])
    if path == "net_grad":
        loss, grad = state["net"].loss_grad(state["features"], state["targets"])
        return {"loss": loss, "grad": grad}
    if path == "stages":
        return _stages(state)
    first, steps = state["step"], case["steps"]
    state["step"] = first + steps
    if path == "ensemble":
        ens = state["ens"]
        ens.step(first, steps)
        return [list(ens.get_state(r)) for r in range(len(ens.params))]
    sim = state["sim"]
    if path == "metrics":
        rows = [_row(*sim.step_diag(s)) for s in range(first, first + steps)]
        x, v = sim.get_state()
        return {"rows": np.array(rows), "x": x, "v": v}
    sim.step(first, steps)
    x, v = sim.get_state()
    if path == "surrogate":
        return {"x": x, "v": v, "counts": sim.surrogate_counts()}
    return {"x": x, "v": v}


def _row(metrics, diag):
    """The driver's metrics row of one step."""
    row = [diag[k] for k in ("meanKinetic", "meanVelocityX", "meanVelocityY", "meanUx", "meanUy", "Qx")]
    for k in ("base", "shifted"):
        row += [diag[k]["occStd"], diag[k]["outBand"], metrics[k]["nParticlesMovedDense"],
                metrics[k]["nParticlesMovedSparse"], metrics[k]["corrRmsDU"], metrics[k]["corrMaxDU"]]
    row += [metrics["closure"][k] for k in ("betaRepairApplied", "meanPdrive", "rmsRepairDU", "maxRepairDU", "rmsEOSDU",
                                            "maxEOSDU")]
    return row


def _stages(state):
    """One step of a program that keeps its state on the host and calls the
    stages one by one, with the benchmark driver's seeds."""
    p, s = state["p"], state["step"]
    state["step"] = s + 1
    x, v = state["x"], state["v"]
    wall = gpu.force_stream_bc(p, x, v, 104729 + 10007 * s)
    cid = gpu.srd_cell_id_with_random_shift(p, x, 130363 + 10007 * s)
    gpu.srd_collision_step(p, v, cid, 433494437 + 10007 * s)
    xr, vr = x.copy(), v.copy()
    zs = 88172645463325252 + 10007 * s
    base, _ = gpu.zone_pass(p, xr, vr, LAYOUT_BASE, zs)
    shifted, _ = gpu.zone_pass(p, xr, vr, LAYOUT_SHIFTED, zs + 4099)
    out = gpu.liquid_closure(p, x, v, xr, vr)
    state["x"], state["v"] = out["x"], out["v"]
    moved = [m[k] for m in (base, shifted) for k in ("nParticlesMovedDense", "nParticlesMovedSparse")]
    return {"x": out["x"], "v": out["v"], "cid": cid, "moved": moved, "pdrive": out["pdrive"],
            "duEOSX": out["duEOSX"], "duEOSY": out["duEOSY"], "nBot": wall["nBot"], "nTop": wall["nTop"]}


# ---- what a pass cannot do without ----

def _net_flops(cells):
    return 2.0 * 9 * cells * sum(a * b for a, b in zip(CHANNELS[:-1], CHANNELS[1:]))


def work(case):
    path = case["path"]
    if path in ("net_forward", "net_grad"):
        cells = case["batch"] * case["Nx"] * case["Ny"]
        if path == "net_forward":
            return {"bytes": cells * (4 + 2) * 4, "flops": _net_flops(cells)}
        # forward, weight gradients, and input gradients of all layers but the first
        flops = 3 * _net_flops(cells) - 2.0 * 9 * cells * CHANNELS[0] * CHANNELS[1]
        return {"bytes": cells * (4 + 2) * 4, "flops": flops}
    if path == "ensemble":
        n = sum(p.n for p in _replicas(case))
        return {"bytes": n * (STEP_BYTES * case["steps"] + STATE_BYTES), "flops": 0}
    cells = case["Nx"] * case["Ny"]
    n = cells * case["ppc"]
    if path == "fields":
        return {"bytes": n * 32 + cells * (4 + 8 * len(FIELDS)), "flops": 0}
    if path == "stages":
        return {"bytes": n * (STEP_BYTES + 4 * STATE_BYTES), "flops": 0}
    flops = _net_flops(cells) * case["steps"] if path == "surrogate" else 0
    return {"bytes": n * (STEP_BYTES * case["steps"] + STATE_BYTES), "flops": flops}


# ---- results in 64 bits ----

def exact(case, seed):
    if case["path"] == "fields":
        return _exact_fields(_params(case), seed)
    if case["path"] == "net_forward":
        f, _ = _samples(case, seed)
        return _forward(case, _weights(), f).cpu().numpy()
    if case["path"] == "net_grad":
        return _exact_grad(case, *_samples(case, seed))
    return None


def _exact_fields(p, seed):
    x, v = [a.cpu().numpy() for a in _particles(p, _generator(seed))]
    dx, dy = p.Lx / p.Nx, p.Ly / p.Ny
    ix = np.clip(np.floor(x[:, 0] / dx).astype(np.int64), 0, p.Nx - 1)
    iy = np.clip(np.floor(x[:, 1] / dy).astype(np.int64), 0, p.Ny - 1)
    c = iy + p.Ny * ix
    N = np.bincount(c, minlength=p.Nc)
    Px, Py = (np.bincount(c, weights=v[:, k], minlength=p.Nc) for k in (0, 1))
    some = np.maximum(N, 1)
    Ux, Uy = Px / some, Py / some
    s2 = np.bincount(c, weights=(v[:, 0] - Ux[c]) ** 2 + (v[:, 1] - Uy[c]) ** 2, minlength=p.Nc)
    T = np.where(N > 1, s2 / np.maximum(2 * (N - 1), 1), 0.0)
    rho = N / (dx * dy)
    Pkin, Pvir = rho * T, p.Kvirial * (rho - _rho_target(p))
    return {"N": N.astype(np.int32), "Ux": Ux, "Uy": Uy, "Px": Px, "Py": Py, "T": T, "rho": rho, "Pkin": Pkin,
            "Pvir": Pvir, "P": Pkin + Pvir, "rhoTarget": np.full(p.Nc, _rho_target(p))}


def _weights(grad=False):
    """The network's layers in 64 bits: W[9 * ci, co] and b[co]."""
    t = torch.tensor(_theta(), dtype=torch.float64, device="cuda")
    out, o = [], 0
    for ci, co in zip(CHANNELS[:-1], CHANNELS[1:]):
        w = t[o:o + co * 9 * ci].reshape(co, 9 * ci).t().contiguous().requires_grad_(grad)
        b = t[o + co * 9 * ci:o + co * 9 * ci + co].clone().requires_grad_(grad)
        o += co * 9 * ci + co
        out.append((w, b))
    return out


def _forward(case, layers, features):
    """x periodic, zeros beyond the walls in y; taps in (dx, dy) order."""
    a = torch.tensor(features, dtype=torch.float64, device="cuda").reshape(case["batch"], case["Nx"], case["Ny"], -1)
    for li, (w, b) in enumerate(layers):
        rows = torch.cat([a[:, -1:], a, a[:, :1]], dim=1)
        pad = torch.nn.functional.pad(rows, (0, 0, 1, 1))
        taps = [pad[:, dx:dx + case["Nx"], dy:dy + case["Ny"]] for dx in range(3) for dy in range(3)]
        a = torch.cat(taps, dim=-1).reshape(-1, w.shape[0]) @ w + b
        if li < len(layers) - 1:
            a = torch.relu(a)
        a = a.reshape(case["batch"], case["Nx"], case["Ny"], -1)
    return a.reshape(case["batch"], case["Nx"] * case["Ny"], -1)


def _exact_grad(case, features, targets):
    layers = _weights(grad=True)
    out = _forward(case, layers, features)
    loss = ((out - torch.tensor(targets, dtype=torch.float64, device="cuda")) ** 2).mean()
    loss.backward()
    grad = torch.cat([g for w, b in layers for g in (w.grad.t().reshape(-1), b.grad)])
    return {"loss": float(loss.detach()), "grad": grad.cpu().numpy()}
