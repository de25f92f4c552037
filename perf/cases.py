"""The work that programs hand to this framework, as timed cases.

Every case is a call sequence through the public classes (`Model`, `Ensemble`, `Mlp`): a model of
a synthetic catchment stepped over real forcing, with the results read back, or the learned warm
start's network trained and evaluated. The catchment belongs to the case (a program steps one
basin); the seed gives the weather and the state the run starts from.

A model starts from a warm state, as a run continued from a state file does: discharge follows
the upstream area, the soil holds water, and part of the catchment has snow. The forcing frames
are consecutive hours (days) of the synthetic weather, taken in turn by the passes.
"""

import functools
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "wflow.jl_amd"))

from wflowhip import Ensemble, Mlp, Model, Var, _abi, synth  # noqa: E402

NODE_ORDER = _abi.WFH_MEM_DEVICE_NODE_ORDER

# The states a program keeps or writes after a step
STATES = (Var.SATWATERDEPTH, Var.USTORELAYERDEPTH, Var.CANOPY_STORAGE, Var.SNOW_STORAGE, Var.SNOW_WATER,
          Var.SSF_Q, Var.LAND_Q, Var.LAND_H, Var.RIVER_Q, Var.RIVER_H)


def _model(name, nx, ny, steps, **options):
    """A model case: grid nx x ny, `steps` time steps a pass, and the options that differ from
    the plain hourly model with forcing on the device in node order."""
    case = {"name": name, "kind": "model", "nx": nx, "ny": ny, "steps": steps, "dt": 3600.0, "cell": 250.0,
            "river": 500, "forcing": "node", "members": 1, "graph": False, "adaptive": False, "snow_transport": False,
            "reservoirs": 0, "floodplain": False, "balance": True, "terrain": 1}
    case.update(options)
    return case


def listed():
    return [
        # a small study basin over one day: every hour's discharge is read as it is computed, so
        # the latency of a step, its launches and its read-backs count
        _model("small_basin_day", 61, 67, 24, river=20, forcing="device", read_each=True),
        # a regional basin over half a day, forcing resident on the GPU
        _model("regional_500", 509, 487, 12, river=120),
        # the same kind of basin with forcing handed over from host arrays every hour, as a
        # program that reads weather files does
        _model("host_forcing_1000", 1021, 997, 4, river=300, forcing="host"),
        # a large country grid, the benchmark's own size and hourly step
        _model("country_4096", 4096, 4096, 2, river=2000),
        # the reference's most common set-up: daily steps, here 24 land and 96 river sub-steps
        _model("daily_256", 256, 256, 2, river=100, dt=86400.0, cell=1000.0),
        # many catchments of different size stepped as one model from a captured graph
        _model("batch_24", 300, 300, 4, river=100, cell=1000.0, members=24, graph=True),
        # sub-steps chosen by the Courant condition
        _model("adaptive_250", 251, 247, 1, river=100, adaptive=True),
        # a floodplain on every river cell
        _model("floodplain_500", 509, 503, 2, river=150, floodplain=True),
        # a mountain basin with lateral snow transport and reservoirs of all outflow types
        _model("reservoirs_snow_800", 797, 811, 3, river=250, reservoirs=24, snow_transport=True, forcing="device"),
        # a parameter ensemble (calibration, uncertainty) of one basin
        {"name": "ensemble_128x256", "kind": "ensemble", "nx": 257, "ny": 251, "members": 128, "steps": 3, "dt": 3600.0,
         "cell": 250.0, "river": 100, "terrain": 1},
        # one training epoch of the warm-start network on harvested rows
        {"name": "network_epoch", "kind": "train", "rows": 300_000, "batch": 8192},
        # the network's proposals for a batch of solves
        {"name": "network_predict", "kind": "predict", "rows": 1_000_003},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["plain", "plain", "plain", "plain", "host", "daily", "daily", "batch", "batch", "adaptive",
                       "floodplain", "reservoirs", "reservoirs", "ensemble", "ensemble", "train", "predict"])
    terrain = rng.randrange(1, 1000)

    def grid(lo, hi):
        side = _log_int(rng, lo, hi)
        return side, max(lo, int(side * rng.uniform(0.8, 1.25)))

    def threshold(nx, ny):
        return max(20, int(nx * ny / rng.uniform(1500.0, 8000.0) * min(1.0, 512.0 / nx)))

    if kind == "train":
        return {"kind": "train", "rows": _log_int(rng, 20_000, 1_000_000), "batch": rng.choice([2048, 8192, 16384])}
    if kind == "predict":
        return {"kind": "predict", "rows": _log_int(rng, 1_000, 4_000_000)}
    if kind == "ensemble":
        members = rng.choice([64, 128, 256])
        nx, ny = grid(60, 300 if members < 256 else 200)
        return {"kind": "ensemble", "nx": nx, "ny": ny, "members": members, "steps": rng.randrange(1, 5), "dt": 3600.0,
                "cell": 250.0, "river": threshold(nx, ny), "terrain": terrain}
    lo, hi = {"plain": (40, 1800), "host": (100, 1200), "daily": (40, 400), "batch": (60, 400), "adaptive": (60, 300),
              "floodplain": (60, 600), "reservoirs": (200, 1000)}[kind]
    nx, ny = grid(lo, hi)
    steps = max(1, min(24, int(2e6 / (nx * ny))))
    options = {"river": threshold(nx, ny), "terrain": terrain, "balance": rng.random() < 0.7}
    if kind == "plain":
        options.update(forcing=rng.choice(["node", "device"]), graph=rng.random() < 0.3)
    elif kind == "host":
        options.update(forcing="host")
    elif kind == "daily":
        options.update(dt=86400.0, cell=1000.0)
        steps = min(steps, 4)
    elif kind == "batch":
        options.update(members=rng.randrange(2, 30), cell=1000.0, graph=rng.random() < 0.5)
        steps = min(steps, 6)
    elif kind == "adaptive":
        options.update(adaptive=True)
        steps = 1
    elif kind == "floodplain":
        options.update(floodplain=True)
        steps = min(steps, 4)
    else:
        options.update(reservoirs=rng.randrange(4, 30), snow_transport=rng.random() < 0.6)
        steps = min(steps, 4)
    case = _model("", nx, ny, steps, **options)
    del case["name"]
    return case


# ---- catchments -----------------------------------------------------------------------------

@functools.lru_cache(maxsize=2)
def _catchment(nx, ny, cell, dt, river, members, reservoirs, floodplain, terrain):
    """The static maps of a case's basin, or of its `members` basins stacked as one model (their
    sides between half and one and a half times the case's)."""
    if members > 1:
        rng = np.random.default_rng(terrain)
        scale = np.exp(rng.uniform(math.log(0.5), math.log(1.5), (members, 2)))
        parts = [synth.make_catchment(max(16, int(nx * a)), max(16, int(ny * b)), cell=cell, dt=dt,
                                      river_threshold=river, seed=1000 * terrain + k)
                 for k, (a, b) in enumerate(scale)]
        c = synth.make_batch(parts)
        c.upstream_area = np.concatenate([p.upstream_area for p in parts])
    else:
        c = synth.make_catchment(nx, ny, cell=cell, dt=dt, river_threshold=river, seed=terrain)
    if reservoirs:
        synth.add_reservoirs(c, reservoirs, seed=terrain, radius=2, curves=True)
    if floodplain:
        synth.add_floodplain(c, seed=terrain)
    return c


def _basin(case):
    return _catchment(case["nx"], case["ny"], case["cell"], case["dt"], case["river"],
                      case.get("members", 1) if case["kind"] == "model" else 1, case.get("reservoirs", 0),
                      case.get("floodplain", False), case["terrain"])


def _frames(c, case, seed, node):
    """Forcing frames (precipitation, potential evaporation, temperature), consecutive time steps
    from a start in the year that the seed gives; on the GPU, in land order or in node order."""
    count = 4 if c.n > 4_000_000 else 24
    first = (seed % 300) * 24 + 6 if case["dt"] < 86400.0 else seed % 300
    elev = torch.as_tensor(c.arrays["elevation"], device="cuda")
    if node is not None:
        elev = elev[node].contiguous()
    return [synth.forcing_torch(c, first + k, elev, seed=seed) for k in range(count)]


# ---- preparation ----------------------------------------------------------------------------

def _warm_state(m, c, seed):
    """A state as a run continued from a state file has it."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    rand = functools.partial(torch.rand, generator=g, device="cuda", dtype=torch.float64)
    A = c.arrays
    n = c.n
    dev = functools.partial(torch.as_tensor, device="cuda")
    runoff = float(np.random.default_rng(seed).uniform(0.2, 0.8)) * 1e-3 / 86400.0  # m/s over the upstream area
    riv = dev(A["river_location"]).bool()
    q = dev(c.upstream_area)[riv].double() * (c.cell * c.cell * runoff)
    slope = dev(A["river_slope"]).clamp(min=1e-5)
    width = dev(A["river_width"])
    # uniform flow in a wide channel: h = (n q / (w sqrt(s)))^(3/5)
    h = (dev(A["river_manning_n"]) * q / (width * slope.sqrt())) ** 0.6
    m.set_value(Var.RIVER_Q, q.cpu().numpy())
    m.set_value(Var.RIVER_H, h.cpu().numpy())
    pore = (dev(A["theta_s"]) - dev(A["theta_r"])) * dev(A["soil_thickness"])
    m.set_value_device(Var.SATWATERDEPTH, (pore * (0.7 + 0.2 * rand(n))).contiguous())
    m.set_value_device(Var.SNOW_STORAGE, (0.05 * rand(n) * (rand(n) < 0.3)).contiguous())
    m.set_value_device(Var.CANOPY_STORAGE, (dev(A["max_canopy_storage"]) * rand(n)).contiguous())
    torch.cuda.synchronize()


def _prepare_model(case, seed):
    c = _basin(case)
    m = Model(c, water_mass_balance=case["balance"], adaptive=case["adaptive"], snow_transport=case["snow_transport"])
    _warm_state(m, c, seed)
    node = torch.as_tensor(m.node_order(), device="cuda") if case["forcing"] == "node" else None
    frames = _frames(c, case, seed, node)
    if case["forcing"] == "host":
        frames = [tuple(f.cpu().numpy() for f in fr) for fr in frames]
    if case["reservoirs"]:
        m.set_julian_day(1 + seed % 365)
    if case["graph"]:
        m.set_graph()
    out = {v.name.lower(): torch.empty(_abi.var_count(v, c.n, c.nriv, c.nlayers, c.nres), dtype=torch.float64,
                                       device="cuda") for v in STATES}
    out["discharge"] = torch.empty((case["steps"], c.nriv), dtype=torch.float64, device="cuda")
    if case["reservoirs"]:
        out["reservoir_storage"] = torch.empty(c.nres, dtype=torch.float64, device="cuda")
    if case["floodplain"]:
        out["floodplain_storage"] = torch.empty(c.nriv, dtype=torch.float64, device="cuda")
    return {"case": case, "model": m, "frames": frames, "next": 0, "out": out,
            "kind": NODE_ORDER if case["forcing"] == "node" else None}


def _factors(members, seed):
    rng = np.random.default_rng(seed)
    return [np.concatenate([[1.0], np.exp(0.3 * rng.standard_normal(members - 1))]) for _ in range(3)]


def _prepare_ensemble(case, seed):
    c = _basin(case)
    ens = Ensemble(c, *_factors(case["members"], seed))
    return {"case": case, "model": ens, "frames": _frames(c, case, seed, None), "next": 0}


def _rows(count, seed):
    """Features of kinematic-wave solves (logarithms of discharge, geometry and time step, a
    signed logarithm of the lateral inflow, the exponent) with a smooth normalised target."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    scale = torch.tensor([1.6, 1.6, 0.5, 0.1, 0.3, 0.6, 2.0, 0.0], device="cuda")
    shift = torch.tensor([-2.0, -2.0, 0.6, 2.4, 3.2, -1.5, -6.0, 0.6], device="cuda")
    x = torch.randn((count, 8), generator=g, device="cuda") * scale + shift
    t = torch.tanh(0.6 * (x[:, 0] + 2.0)) - 0.3 * (x[:, 1] + 2.0) + 0.1 * torch.randn(count, generator=g, device="cuda")
    return x.contiguous(), ((t - t.mean()) / t.std()).contiguous()


_MEAN = np.array([-2.0, -2.0, 0.6, 2.4, 3.2, -1.5, -6.0, 0.6], np.float32)
_STD = np.array([1.6, 1.6, 0.5, 0.1, 0.3, 0.6, 2.0, 1.0], np.float32)


def _weights(seed):
    """Network parameters of the size that training leaves: W1 [64][8], b1, W2 [64][64], b2, w3, b3."""
    rng = np.random.default_rng(seed)
    return np.concatenate([rng.standard_normal(64 * 8) / math.sqrt(8.0), 0.1 * rng.standard_normal(64),
                           rng.standard_normal(64 * 64) / 8.0, 0.1 * rng.standard_normal(64),
                           rng.standard_normal(64) / 8.0, [0.05]]).astype(np.float32)


def _prepare_network(case, seed):
    x, t = _rows(case["rows"], seed)
    net = Mlp(seed=seed)
    net.set_normalization(_MEAN, _STD, 0.0, 1.0)
    net.set_params(_weights(seed))
    return {"case": case, "net": net, "x": x, "t": t,
            "out": torch.empty(case["rows"], dtype=torch.float32, device="cuda")}


def prepare(case, seed):
    if case["kind"] == "model":
        return _prepare_model(case, seed)
    if case["kind"] == "ensemble":
        return _prepare_ensemble(case, seed)
    return _prepare_network(case, seed)


# ---- one pass -------------------------------------------------------------------------------

def _run_model(s):
    m, case, out = s["model"], s["case"], s["out"]
    frames = s["frames"]
    for k in range(case["steps"]):
        m.set_forcing(*frames[s["next"]], memkind=s["kind"])
        s["next"] = (s["next"] + 1) % len(frames)
        m.update_model()
        if case.get("read_each") or k == case["steps"] - 1:
            m.get_value_device(Var.RIVER_Q_AVERAGE, out["discharge"][k])
    for v in STATES:
        m.get_value_device(v, out[v.name.lower()])
    if case["reservoirs"]:
        m.get_value_device(Var.RESERVOIR_STORAGE, out["reservoir_storage"])
    if case["floodplain"]:
        m.get_value_device(Var.FLOODPLAIN_STORAGE, out["floodplain_storage"])
    if not case.get("read_each"):
        return dict(out, discharge=out["discharge"][case["steps"] - 1])
    return out


def _run_ensemble(s):
    ens, case = s["model"], s["case"]
    for _ in range(case["steps"]):
        ens.run_timestep(*s["frames"][s["next"]])
        s["next"] = (s["next"] + 1) % len(s["frames"])
    # the discharge of some members at every river cell, the states of the first and the last
    out = {f"discharge_{k}": ens.get(Var.RIVER_Q_AVERAGE, k) for k in range(0, case["members"], 16)}
    for k in (0, case["members"] - 1):
        for v in (Var.SATWATERDEPTH, Var.USTORELAYERDEPTH, Var.SSF_Q, Var.LAND_Q, Var.RIVER_Q):
            out[f"{v.name.lower()}_{k}"] = ens.get(v, k)
    return out


def run(state):
    kind = state["case"]["kind"]
    if kind == "model":
        return _run_model(state)
    if kind == "ensemble":
        return _run_ensemble(state)
    net = state["net"]
    if kind == "predict":
        return net.predict(state["x"], state["out"])
    loss = net.train_epoch(state["x"], state["t"], batch=state["case"]["batch"])
    return {"loss": loss, "params": net.params()}


# ---- work and exact values ------------------------------------------------------------------

def work(case):
    """Bytes: each cell's forcing, parameters and states read and its states and fluxes written
    once a time step (900 B per cell of the four-layer model, 259 B per member and cell of an
    ensemble, whose maps are shared), plus the states read back. Operations: about 1500 per cell
    and step, and about 200 per further kinematic-wave sub-step of a cell."""
    kind = case["kind"]
    macs = 64 * 8 + 64 * 64 + 64
    if kind == "train":
        return {"bytes": case["rows"] * 36.0, "flops": case["rows"] * 6.0 * macs}
    if kind == "predict":
        return {"bytes": case["rows"] * 36.0, "flops": case["rows"] * 2.0 * macs}
    cells = case["nx"] * case["ny"] * case["members"]
    if kind == "ensemble":
        return {"bytes": 259.0 * cells * case["steps"], "flops": 1500.0 * cells * case["steps"]}
    if case["members"] > 1:
        cells *= 0.82  # mean area of the members, (mean of exp U(log 0.5, log 1.5))^2
    land = 24.0 if case["dt"] > 3600.0 else 1.0
    return {"bytes": cells * (900.0 * case["steps"] + 2 * 8.0 * 11.0),
            "flops": cells * case["steps"] * (1500.0 + 200.0 * (land - 1.0))}


def exact(case, seed):
    """The network's value in 64 bits. A model's or an ensemble's outputs have none: the step is
    computed in 64 bits throughout and has no form without this repository's code. Neither has a
    training epoch, whose updates follow from the network's own 16-bit gradients."""
    if case["kind"] != "predict":
        return None
    x, _ = _rows(case["rows"], seed)
    p = torch.as_tensor(_weights(seed), device="cuda").double()
    w1, b1, w2, b2, w3, b3 = torch.split(p, [512, 64, 4096, 64, 64, 1])
    z = (x.double() - torch.as_tensor(_MEAN, device="cuda").double()) / torch.as_tensor(_STD, device="cuda").double()
    h = torch.relu(z @ w1.reshape(64, 8).T + b1)
    h = torch.relu(h @ w2.reshape(64, 64).T + b2)
    return h @ w3 + b3
