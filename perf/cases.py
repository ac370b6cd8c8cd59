"""The work a program gives this framework, as cases that can be timed.

Kinds of case (``case["kind"]``):

run         Days of one context through ``Engine.run_days``: a single simulation or a batch of
            them, going on from a state that the program has kept.  A pass puts the kept state
            back into the bound buffers (as the C ABI lets a caller do between steps:
            lp_invalidate), runs the days and syncs, as a scenario branch or a repeated
            replicate does; the first day recounts the carried statistics, the sync writes the
            records back into the agent columns.  ``per_call`` days go into each call (0: all of
            them in one).
components  Days stepped component by component (``Engine.step``, one call per component and
            one for the log), as a simulation with a component of its own does.
rollout     The mean-field rollout of the node-level transmission map (``adjoint.rollout``).
gradient    The rollout and its adjoint, for a given adjoint of the incidence.
fit         Loss and gradient of the mean-field calibration: gravity network, seasonality,
            rollout, weekly Poisson likelihood and back, as a step of ``calib.fit_meanfield``.
gravity     Every simulation's gravity network rebuilt on the device
            (``BatchedSims.set_gravity``), as a calibration generation does.
init        Every agent column drawn on the device (``Engine.init_population``).

A run that starts at a tick ``start`` above 0 starts on a routine-immunisation day (a multiple of
14): the first pass over the agents then brings ri_timer up to that day itself.  Component steps
start on the day after one and end before the next, with a vital-dynamics step on the seventh day.
"""

import math

import numpy as np
import torch

from __graft_entry__ import load_package

load_package()

from laser_polio_amd import adjoint, configs  # noqa: E402
from laser_polio_amd import engine as engmod  # noqa: E402
from laser_polio_amd.batch import build_replicates_device  # noqa: E402
from laser_polio_amd.propertyset import PropertySet  # noqa: E402

# agent columns that a day may change (multipliers and chronically_missed never change)
STATE = ("disease_state", "strain", "exposure_timer", "infection_timer", "paralysis_timer", "potentially_paralyzed",
         "paralyzed", "ipv_protected", "ri_timer", "date_of_birth", "date_of_death", "node_id")
# result rows that a day adds to (every other row is written afresh)
ADDED = ("R", "new_exposed", "new_exposed_by_strain", "sia_new_exposed_by_strain")
ROWS = ("S", "E", "I", "R", "E_by_strain", "I_by_strain", "potentially_paralyzed_count", "paralyzed_count",
        "new_potentially_paralyzed", "new_paralyzed", "pop", "births", "deaths", "new_exposed", "new_exposed_by_strain",
        "ri_vaccinated", "ri_protected", "ri_new_exposed_by_strain", "ipv_vaccinated", "sia_vaccinated", "sia_protected",
        "sia_new_exposed_by_strain")
COLUMNS = STATE + ("acq_risk_multiplier", "daily_infectivity", "chronically_missed")

TAU_E, TAU_I = 3.0, configs.DUR_INF_MEAN      # mean exposure and infectious durations of the workloads
R0 = 14.0


def listed():
    return [
        # the smallest simulation of a test or a notebook: three nodes, RI, 40 days in one call
        {"name": "small run", "kind": "run", "model": "small", "place": 42,
         "scale": 1.0, "nodes": 3, "sims": 1, "start": 14, "days": 40, "per_call": 0},
        # the 14-node workload over its whole year, from the initial infections through the epidemic
        {"name": "spatial year", "kind": "run", "model": "spatial", "place": 42,
         "scale": 1.0, "nodes": 14, "sims": 1, "start": 0, "days": 365, "per_call": 0},
        # the national workload, one year from day 994 (endemic), RI every 14 days and two campaigns
        {"name": "national year", "kind": "run", "model": "national", "place": 42,
         "scale": 1.0, "nodes": 774, "sims": 1, "start": 994, "days": 364, "per_call": 0},
        # replicates of calibration trials batched in one context, the whole year
        {"name": "replicates", "kind": "run", "model": "replicates", "place": 42,
         "scale": 1.0, "nodes": 24, "sims": 64, "start": 0, "days": 365, "per_call": 0},
        # 5000 nodes, three strains, a campaign on day 120, at the population scale the seeds are batched at
        {"name": "continental", "kind": "run", "model": "continental", "place": 42,
         "scale": 0.25, "nodes": 5000, "sims": 1, "start": 0, "days": 150, "per_call": 0},
        # a user's own component in the list: every component stepped by itself
        {"name": "component steps", "kind": "components", "model": "spatial", "place": 42,
         "scale": 1.0, "nodes": 14, "sims": 1, "start": 29, "days": 8},
        # half a year of the mean-field map over the national geography, and its gradient
        {"name": "rollout national", "kind": "rollout", "nodes": 774, "days": 180, "checkpoint": 30},
        {"name": "gradient national", "kind": "gradient", "nodes": 774, "days": 180, "checkpoint": 30},
        # the same for one replicate's geography over a year
        {"name": "gradient replicate", "kind": "gradient", "nodes": 23, "days": 365, "checkpoint": 30},
        # one step of a gradient calibration on the national geography
        {"name": "fit national", "kind": "fit", "nodes": 774, "days": 180, "checkpoint": 30},
        # the networks of a calibration generation
        {"name": "gravity national", "kind": "gravity", "model": "national", "place": 42, "nodes": 774, "sims": 4},
        # the national population drawn on the GPU
        {"name": "init national", "kind": "init", "model": "national", "place": 42,
         "scale": 1.0, "nodes": 774, "sims": 1},
    ]


def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(["run"] * 5 + ["components", "rollout", "gradient", "gradient", "fit", "gravity", "init"])
    if kind in ("rollout", "gradient", "fit"):
        nodes = int(_log_uniform(rng, 3, 1200))
        return {"kind": kind, "nodes": nodes, "days": int(_log_uniform(rng, 28, 365)),
                "checkpoint": 30 if kind == "fit" else rng.choice([30, 30, rng.randint(5, 120)])}
    place = rng.randint(1, 10**6)
    if kind == "gravity":
        if rng.random() < 0.5:
            return {"kind": kind, "model": "replicates", "place": place,
                    "nodes": 24, "sims": int(_log_uniform(rng, 2, 256))}
        return {"kind": kind, "model": "national", "place": place,
                "nodes": int(_log_uniform(rng, 50, 774)), "sims": rng.randint(1, 4)}
    model = rng.choice(["small", "spatial", "national", "replicates", "continental"] if kind == "run"
                       else ["small", "spatial", "national", "replicates"])
    case = {"kind": kind, "model": model, "place": place, "scale": _log_uniform(rng, 0.05, 1.0), "nodes": 14, "sims": 1}
    if model == "small":
        case.update(scale=_log_uniform(rng, 0.2, 6.0), nodes=rng.randint(2, 9))
    elif model == "national":
        case.update(scale=_log_uniform(rng, 0.02, 0.5), nodes=int(_log_uniform(rng, 60, 774)))
    elif model == "replicates":
        case.update(nodes=24, sims=int(_log_uniform(rng, 2, 48)))
    elif model == "continental":
        case.update(scale=_log_uniform(rng, 0.01, 0.12), nodes=int(_log_uniform(rng, 1200, 5000)))
    if kind == "init":
        return case
    if kind == "components":
        case["scale"] = min(case["scale"], 0.1 if model in ("national", "replicates") else 1.0)
        case.update(start=14 * rng.randint(1, 6) + 1, days=rng.randint(3, 9))
        return case
    case.update(start=0 if model in ("spatial", "replicates", "continental") else 14 * rng.randint(1, 40),
                days=rng.randint(20, 200))
    case["per_call"] = rng.choice([0, 0, 1, 7])
    return case


# -- simulations -----------------------------------------------------------------------------------
def _small_pars(case, rng, dur):
    """The three-node simulation of the smoke test, to `nodes` nodes, its default options (default
    age pyramid, gamma infectivity, Poisson exposure), RI in every node."""
    n = case["nodes"]
    pop = np.maximum(1000, (np.array([30000, 20000, 15000])[np.arange(n) % 3] * case["scale"]).astype(np.int64))
    d = np.triu(rng.uniform(40, 120, (n, n)), 1)
    return PropertySet({
        "dur": dur, "init_pop": pop, "cbr": np.full(n, 35.0), "r0": 14,
        "r0_scalars": rng.uniform(0.8, 1.2, n), "init_immun": np.full(n, 0.6).tolist(),
        "init_prev": [20] + [0] * (n - 1), "distances": d + d.T, "migration_method": "gravity", "gravity_k": 0.5,
        "max_migr_frac": 0.3, "vx_prob_ri": 0.5, "stop_if_no_cases": False, "verbose": 0})


def _pars_list(case, seed, dur):
    """The case's simulations: a geography is a configuration of its own (`place`), the seed draws
    the population, the infections and every day's events in it."""
    model, scale, place = case["model"], case.get("scale", 1.0), case["place"]
    rng = np.random.default_rng([seed, 11])
    if model == "small":
        plist = [_small_pars(case, np.random.default_rng([place, 7]), dur)]
    elif model == "spatial":
        plist = [configs.spatial14_pars(scale=scale, seed=place, dur=dur)]
    elif model == "national":
        plist = [configs.nigeria_national_pars(scale=scale, seed=place + k, dur=dur, n=case["nodes"])
                 for k in range(case["sims"])]
    elif model == "continental":
        plist = [configs.continental_pars(scale=scale, seed=place, dur=dur, n=case["nodes"])]
    else:
        plist = [configs.replicate_pars(i, master_seed=place, scale=scale, dur=dur) for i in range(case["sims"])]
    for pars in plist:
        pars["seed"] = int(rng.integers(1, 2**31))
    return plist


def _context(case, seed, dur):
    """A batch of the case's simulations, its context on the GPU with the population drawn there."""
    batch = build_replicates_device(_pars_list(case, seed, dur), configs.build)
    return batch, batch.prepare()


def _keep(batch, eng, case):
    """The program's own stream and its copy of the state at the start tick."""
    stream = torch.cuda.Stream()
    eng.set_stream(stream)
    if case["start"] > 0:
        eng.run_days(0, case["start"])
        eng.sync()
    names = STATE + ("live_end",) + ADDED
    kept = [(eng.tensors[n], eng.tensors[n].clone()) for n in names]
    torch.cuda.synchronize()
    return {"batch": batch, "eng": eng, "stream": stream, "kept": kept}


def _restore(state):
    """The kept state back into the bound buffers; the next day recounts from them."""
    with torch.cuda.stream(state["stream"]):
        for bound, saved in state["kept"]:
            bound.copy_(saved)
    eng = state["eng"]
    if eng.lib.lp_invalidate(eng.ctx) != 0:
        raise engmod.LPError("lp_invalidate")


def _outputs(eng):
    out = {n: eng.tensors[n] for n in STATE + ("live_end",)}
    out.update({"row " + n: eng.tensors[n] for n in ROWS})
    return out


# -- mean-field inputs ---------------------------------------------------------------------------------
def _meanfield_inputs(case, seed):
    """Geography, compartments and parameters of a mean-field problem, float64 on the host: the
    national geography's populations, distances, immunity and parameters for `nodes` nodes."""
    rng = np.random.default_rng([seed, 5])
    n, T = case["nodes"], case["days"]
    pop = np.round(rng.lognormal(np.log(2.5e5), 0.6, n))
    xy = rng.uniform(0, 1000, (n, 2))
    d = np.sqrt(((xy[:, None, :] - xy[None, :, :]) ** 2).sum(-1))
    S = np.round(pop * rng.uniform(0.2, 0.3, n))
    I = np.where(np.arange(n) == 0, np.round(0.005 * pop), np.round(rng.uniform(0, 20, n)))
    E = np.round(I * rng.uniform(0.0, 0.3, n))
    x = {"pop": pop, "dist": d, "S": S, "E": E, "I": I, "rho": rng.uniform(0.9, 1.1, n), "inv_pop": 1.0 / pop,
         "r0s": rng.lognormal(0.0, 0.3, n), "k": 0.5 * rng.uniform(0.6, 1.4), "a": 1.0, "b": 1.0, "c": 2.0,
         "amp": 0.4 * rng.uniform(0.6, 1.2), "peak": 180.0, "doy": 1.0 + np.arange(1, T + 1) % 365,
         "diy": np.full(T, 365.0), "g_inc": rng.standard_normal((T, n)) / (n * T),
         "y": rng.poisson(40.0, (T, n)).astype(np.float64)}
    # what every float32 reader of these inputs holds
    return {k: np.asarray(v, dtype=np.float32).astype(np.float64) for k, v in x.items()}


IOTA = R0 / TAU_I
FIT = ("r0s", "k", "a", "b", "c", "amp", "peak")


def _gravity64(pop, dist, k, a, b, c, max_frac):
    """Row-capped gravity network in plain torch, any floating type."""
    n = pop.shape[0]
    off = ~torch.eye(n, dtype=torch.bool, device=pop.device)
    net = k * pop[:, None] ** a * pop[None, :] ** b / torch.where(off, dist, torch.ones_like(dist)) ** c
    net = torch.where(off, net, torch.zeros_like(net)) / pop.sum() ** c
    rs = net.sum(dim=1, keepdim=True)
    return net * torch.where(rs > max_frac, max_frac / rs, torch.ones_like(rs))


def _rollout64(r0s, net, season, S, E, I, rho, inv_pop, iota, ite, iti):
    keep = 1.0 - net.sum(dim=1)
    out = []
    for t in range(season.shape[0]):
        m = iota * (I * keep + net.t() @ I)
        lam = rho * S * (-torch.expm1(-(m * season[t] * r0s * inv_pop)))
        S, E, I = S - lam, E + lam - E * ite, I + E * ite - I * iti
        out.append(lam)
    return torch.stack(out)


# -- the case functions ------------------------------------------------------------------------------------
def prepare(case, seed):
    kind = case["kind"]
    if kind in ("run", "components"):
        batch, eng = _context(case, seed, case["start"] + case["days"])
        return {"case": case, **_keep(batch, eng, case)}
    if kind == "init":
        batch, eng = _context(case, seed, 30)
        specs, infected = batch.device_init
        slots = np.concatenate([np.asarray(s, np.int64) + o for s, o in zip(infected, batch.slot_off)])
        return {"case": case, "batch": batch, "eng": eng, "specs": specs, "slots": slots}
    if kind == "gravity":
        batch, eng = _context({**case, "scale": 0.002}, seed, 30)
        rng = np.random.default_rng([seed, 3])
        S = case["sims"]
        new = {"k": rng.uniform(0.1, 1.0, S), "a": rng.uniform(0.8, 1.2, S), "b": rng.uniform(0.8, 1.2, S),
               "c": rng.uniform(1.5, 2.5, S), "max_rowsum": rng.uniform(0.05, 0.3, S)}
        batch.set_gravity(pull=False)      # the program's populations and distances on the device
        return {"case": case, "batch": batch, "eng": eng, "new": new}
    x = _meanfield_inputs(case, seed)
    dev = torch.device("cuda", torch.cuda.current_device())
    t = {k: torch.as_tensor(v, dtype=torch.float32, device=dev) for k, v in x.items()}
    state = {"case": case, "t": t}
    if kind == "fit":
        state["y"] = adjoint.weekly(t["y"])
        state["params"] = {k: t[k].clone().requires_grad_(True) for k in FIT}
    else:
        x64 = {k: torch.as_tensor(v) for k, v in x.items()}
        net = _gravity64(x64["pop"], x64["dist"], x64["k"], x64["a"], x64["b"], x64["c"], 0.3).to(torch.float32)
        season = 1.0 + x64["amp"] * torch.cos(2.0 * np.pi * (x64["doy"] - x64["peak"]) / x64["diy"])
        state["net"], state["season"] = net.to(dev), season.to(torch.float32).to(dev)
        if kind == "gradient":
            names = ("r0s", "net", "season", "S", "E", "I")
            src = {**t, "net": state["net"], "season": state["season"]}
            state["leaves"] = [src[k].clone().requires_grad_(True) for k in names]
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "run":
        eng, t, end = state["eng"], case["start"], case["start"] + case["days"]
        _restore(state)
        step = case["per_call"] or case["days"]
        while t < end:
            eng.run_days(t, min(end, t + step))
            t += step
        eng.sync()
        return _outputs(eng)
    if kind == "components":
        eng, batch = state["eng"], state["batch"]
        _restore(state)
        stages = [engmod.STAGE_VITAL, engmod.STAGE_DISEASE]
        if case["model"] in ("small", "national"):
            stages.append(engmod.STAGE_RI)
        if batch.cfg.n_sia_events:
            stages.append(engmod.STAGE_SIA)
        for t in range(case["start"], case["start"] + case["days"]):
            for stage in stages + [engmod.STAGE_TRANSMISSION, engmod.STAGE_LOG]:
                eng.step(t, stage)
        eng.sync()
        return _outputs(eng)
    if kind == "init":
        eng = state["eng"]
        eng.init_population(state["specs"], state["slots"])
        return {n: eng.tensors[n] for n in COLUMNS}
    if kind == "gravity":
        state["batch"].set_gravity(pull=False, **state["new"])
        return {n: state["eng"].tensors[n] for n in ("network_t", "keep")}
    t = state["t"]
    if kind == "fit":
        p = state["params"]
        for v in p.values():
            v.grad = None
        net = adjoint.gravity_network(t["pop"], t["dist"], p["k"], p["a"], p["b"], p["c"], 0.3)
        season = adjoint.seasonality(p["amp"], p["peak"], t["doy"], t["diy"])
        inc = adjoint.rollout(p["r0s"], net, season, t["S"], t["E"], t["I"], t["rho"], t["inv_pop"], IOTA,
                              1.0 / TAU_E, 1.0 / TAU_I)
        loss = adjoint.poisson_nll(adjoint.weekly(inc), state["y"])
        loss.backward()
        return {"loss": loss.detach(), "inc": inc.detach(), "grad": [p[k].grad for k in FIT]}
    if kind == "rollout":
        with torch.no_grad():
            return adjoint.rollout(t["r0s"], state["net"], state["season"], t["S"], t["E"], t["I"], t["rho"],
                                   t["inv_pop"], IOTA, 1.0 / TAU_E, 1.0 / TAU_I, case["checkpoint"])
    r0s, net, season, S, E, I = state["leaves"]
    for v in state["leaves"]:
        v.grad = None
    inc = adjoint.rollout(r0s, net, season, S, E, I, t["rho"], t["inv_pop"], IOTA, 1.0 / TAU_E, 1.0 / TAU_I,
                          case["checkpoint"])
    inc.backward(t["g_inc"])
    return {"inc": inc.detach(), "grad": [v.grad for v in state["leaves"]]}


def _agents(case):
    """Agents of the case's simulations, about."""
    model, n, s, scale = case["model"], case["nodes"], case["sims"], case.get("scale", 0.002)
    if model == "small":
        return n * 21700.0 * scale
    if model == "spatial":
        return 14 * 3.4e5 * scale
    if model == "national":
        return n * s * 2.95e5 * scale
    if model == "continental":
        return n * 2.72e5 * scale
    return s * 3.25e6 * scale


def work(case):
    kind = case["kind"]
    if kind in ("run", "components"):
        # every agent column read once (32 B), those that change written once (23 B); the result
        # rows (22 arrays, 6 of them by strain) and the network's contraction of each day
        n = case["nodes"] * case["sims"]
        net = case["nodes"] * n
        return {"bytes": _agents(case) * 55.0 + case["days"] * n * 4.0 * (16 + 6 * 3) + 4.0 * net,
                "flops": case["days"] * 2.0 * 3 * net}
    if kind == "init":
        return {"bytes": _agents(case) * 1.3 * 32.0, "flops": 0.0}
    if kind == "gravity":
        return {"bytes": 12.0 * case["nodes"] ** 2 * case["sims"], "flops": 0.0}
    n, T = float(case["nodes"]), float(case["days"])
    if kind == "rollout":
        return {"bytes": 4.0 * (n * n + T * n + 8 * n), "flops": 2.0 * n * n * T}
    # forward and backward matrix-vector products and the network's adjoint
    reads = 2.0 if kind == "fit" else 3.0
    return {"bytes": 4.0 * (reads * n * n + 2 * T * n + 14 * n), "flops": 6.0 * n * n * T}


def exact(case, seed):
    """What the floating outputs are in 64 bits, in plain torch; the days of simulations have whole
    outputs only, and the drawn population has no value of its own."""
    kind = case["kind"]
    if kind in ("run", "components", "init"):
        return None
    dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
    f64 = dict(dtype=torch.float64, device=dev)
    if kind == "gravity":
        rng = np.random.default_rng([seed, 3])
        S = case["sims"]
        k, a, b = rng.uniform(0.1, 1.0, S), rng.uniform(0.8, 1.2, S), rng.uniform(0.8, 1.2, S)
        c, top = rng.uniform(1.5, 2.5, S), rng.uniform(0.05, 0.3, S)
        nets, keeps = [], []
        for s, pars in enumerate(_pars_list({**case, "scale": 0.002}, seed, 30)):
            net = _gravity64(torch.as_tensor(np.asarray(pars.init_pop, np.float64), **f64),
                             torch.as_tensor(pars.distances, **f64), float(k[s]), float(a[s]), float(b[s]), float(c[s]),
                             float(top[s]))
            nets.append(net.t().reshape(-1).cpu())
            keeps.append((1.0 - net.sum(dim=1)).cpu())
        return {"network_t": torch.cat(nets), "keep": torch.cat(keeps)}
    x = {k: torch.as_tensor(v, **f64) for k, v in _meanfield_inputs(case, seed).items()}
    consts = (x["rho"], x["inv_pop"], IOTA, 1.0 / TAU_E, 1.0 / TAU_I)
    if kind == "fit":
        p = {k: x[k].clone().requires_grad_(True) for k in FIT}
        net = _gravity64(x["pop"], x["dist"], p["k"], p["a"], p["b"], p["c"], 0.3)
        season = 1.0 + p["amp"] * torch.cos(2.0 * np.pi * (x["doy"] - p["peak"]) / x["diy"])
        inc = _rollout64(p["r0s"], net, season, x["S"], x["E"], x["I"], *consts)
        weeks = inc.shape[0] // 7
        mu, y = (v[:7 * weeks].reshape(weeks, 7, -1).sum(dim=1) for v in (inc, x["y"]))
        loss = (mu - y * torch.log(mu + 1e-12)).sum()
        loss.backward()
        return {"loss": loss.detach(), "inc": inc.detach(), "grad": [p[k].grad for k in FIT]}
    net = _gravity64(*(torch.as_tensor(x[k].cpu()) for k in ("pop", "dist", "k", "a", "b", "c")), 0.3)
    net = net.to(torch.float32).to(**f64)      # the float32 network and season that the call is given
    season = (1.0 + x["amp"] * torch.cos(2.0 * np.pi * (x["doy"] - x["peak"]) / x["diy"])).to(torch.float32).to(**f64)
    leaves = [x["r0s"], net, season, x["S"], x["E"], x["I"]]
    if kind == "rollout":
        return _rollout64(*leaves, *consts)
    leaves = [v.clone().requires_grad_(True) for v in leaves]
    inc = _rollout64(*leaves, *consts)
    inc.backward(x["g_inc"])
    return {"inc": inc.detach(), "grad": [v.grad for v in leaves]}
