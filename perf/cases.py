"""The work a user of this framework has it do, as timed cases.

Each case is one call sequence of an inference or prediction program through
the package's public entry points: an ABC-SMC generation, an MC3 update by
model-based proposals, one sweep of an uneven batch, a PMCMC likelihood
estimate, the observation model over many samples, posterior samples loaded
from host arrays, ABC-SMC importance weights, and prediction requests.  Model
structures and sizes are those of beep_amd.configs and beep_amd.serving.

`prepare` builds what such a program holds before the call (contexts with
their models, parameter vectors, current chains), `run` makes the call.  A
model's structure and sizes depend on the case only; parameters, keys, chains
and counts come from the seed.
"""
import functools
import math

import numpy as np

from beep_amd import _lib, batch, configs, serving, spec as specmod


def listed():
    return [
        # One particle of the single-area SEIR model: the smallest call, where an
        # interactive user or a plain sampler pays the launch and the step latency.
        {"name": "seir_one", "kind": "generation", "model": "seir", "areas": 1, "groups": 1, "days": 100, "n": 1},
        # A generation of the single-area model: many tiny instances.
        {"name": "seir_generation", "kind": "generation", "model": "seir", "areas": 1, "groups": 1, "days": 100,
         "n": 4096},
        # The 100-area, 4-age-group spatial ABC-SMC generation at its configured size.
        {"name": "spatial_generation", "kind": "generation", "model": "spatial", "areas": 100, "groups": 4, "days": 200,
         "n": 4096},
        # MC3 on the spatial model: every chain's MBP proposal, likelihood and acceptance.
        {"name": "spatial_proposals", "kind": "proposals", "model": "spatial", "areas": 100, "groups": 4, "days": 200,
         "n": 256, "mask": 0.0},
        # Fixed-tree / slice-time proposals on an odd-sized nine-group model: masked MBPs of few chains.
        {"name": "masked_proposals", "kind": "proposals", "model": "areas", "areas": 37, "groups": 9, "days": 151,
         "n": 24, "mask": 0.3},
        # One sweep over many model sizes at once (areas 10-400, horizons 50-400, 1/4/9 groups).
        {"name": "uneven_sweep", "kind": "batch", "models": 20, "particles": 48, "ladders": 20},
        # The particle-filter likelihood of the dense-mixing 317-area, 9-group model.
        {"name": "dense_filter", "kind": "filter", "model": "dense", "areas": 317, "groups": 9, "days": 300,
         "section": 30, "n": 512},
        # A particle filter on an ordinary sparse model, in fortnights.
        {"name": "sparse_filter", "kind": "filter", "model": "areas", "areas": 25, "groups": 4, "days": 112,
         "section": 14, "n": 500},
        # Error functions per data table of a set of simulated samples.
        {"name": "table_errors", "kind": "tables", "model": "spatial", "areas": 100, "groups": 4, "days": 200, "n": 512},
        # Posterior samples loaded from host arrays, replayed, scored and read back.
        {"name": "sample_load", "kind": "load", "areas": 100, "days": 200, "n": 6},
        # Importance weights of an ABC-SMC generation of the spatial model (22 parameters).
        {"name": "abcsmc_weights", "kind": "weights", "particles": 4096, "variables": 22},
        # A burst of prediction requests over the serving catalogue.
        {"name": "serving_burst", "kind": "serving", "requests": 10, "posterior": 1000},
    ]


def draw(rng):
    def logint(lo, hi):
        return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))

    kind = rng.choice(["generation", "generation", "generation", "proposals", "proposals", "batch", "filter", "filter",
                       "tables", "load", "weights", "serving"])
    if kind in ("generation", "proposals"):
        model = rng.choice(["seir", "spatial", "areas"] if kind == "generation" else ["spatial", "areas"])
        if model == "seir":
            return {"kind": kind, "model": model, "areas": 1, "groups": 1, "days": rng.randint(40, 200),
                    "n": logint(1, 4096)}
        groups = 4 if model == "spatial" else rng.choice([1, 4, 9])
        case = {"kind": kind, "model": model, "areas": rng.randint(11, 100), "groups": groups,
                "days": rng.randint(50, 200), "n": logint(16, 2048) if kind == "generation" else logint(8, 256)}
        if kind == "proposals":
            case["mask"] = rng.choice([0.0, 0.0, 0.3, 1.0])
        return case
    if kind == "batch":
        return {"kind": kind, "models": rng.randint(4, 20), "particles": rng.randint(8, 48), "ladders": rng.randint(4, 20)}
    if kind == "filter":
        if rng.random() < 0.4:
            return {"kind": kind, "model": "dense", "areas": rng.randint(64, 317), "groups": 9,
                    "days": rng.randint(60, 300), "section": rng.choice([14, 30]), "n": logint(64, 512)}
        return {"kind": kind, "model": "areas", "areas": rng.randint(11, 60), "groups": rng.choice([1, 4]),
                "days": rng.randint(56, 200), "section": rng.choice([7, 14, 28]), "n": logint(50, 1000)}
    if kind == "tables":
        return {"kind": kind, "model": "spatial", "areas": rng.randint(20, 100), "groups": 4, "days": rng.randint(60, 200),
                "n": logint(8, 512)}
    if kind == "load":
        return {"kind": kind, "areas": rng.randint(11, 100), "days": rng.randint(50, 200), "n": rng.randint(1, 6)}
    if kind == "weights":
        return {"kind": kind, "particles": logint(200, 4096), "variables": rng.randint(2, 22)}
    return {"kind": kind, "requests": rng.randint(3, 10), "posterior": rng.randint(400, 1000)}


# ---- models: a function of the sizes alone ----

@functools.lru_cache(maxsize=None)
def _model(model, areas, groups, days, section=0):
    """(spec, true parameters) of a case's model; with `section`, a model for
    the particle filter: observations of one simulation at the true
    parameters, in sections of that many days."""
    if model == "seir":
        return configs.seir_single(period=days)
    if model == "spatial":
        return configs.spatial_abcsmc(A=areas, period=days)
    if model == "dense":
        spec, truth = configs.dense_pmcmc(A=areas, period=days, with_obs=False)
        tr = 6
    else:
        spec, truth = configs.seir_areas(areas, groups, days, seed=31 + areas, daily_obs=not section)
        tr = 2
    if section:
        one = _lib.Context(spec, capacity=1, nslot=1, keep=_lib.KEEP_TRANSNUM)
        one.set_param([0], truth[None, :])
        one.simulate([0], [0], [123456], seed=17, stream=1)
        counts = one.get_transnum(0)
        one.close()
        if model == "dense":
            spec["obs"] = configs.daily_observations(counts, tr=tr)
        else:
            y = counts[:, :, tr, :].sum(-1)                    # [day][area]
            spec["obs"] = [{"y": float(y[d, c]), "sd": max(5.0, 0.1 * float(y[d, c])), "type": "normal", "datatable": 0,
                            "graph": c, "sett_i": d, "sett_f": d + 1, "area": [c], "dp": list(range(groups)), "tr": [tr]}
                           for c in range(areas) for d in range(days)]
        spec["sections"] = [(a, min(days, a + section)) for a in range(0, days, section)]
    return spec, truth


def _case_model(case):
    return _model(case["model"], case["areas"], case["groups"], case["days"], case.get("section", 0))


def _dims(spec):
    return spec["A"], spec["G"], len(spec["comps"]), len(spec["trans"]), specmod.nsteps(spec)


def _batch_workload(case):
    """Models of the uneven batch: areas 10-400, horizons 50-400, 1, 4 or 9
    groups; ABC-SMC groups of `particles` and MC3 ladders of 8 chains."""
    rng = np.random.default_rng(1000 * case["models"] + 10 * case["ladders"] + case["particles"])

    def sizes(k):
        return rng.integers(10, 401, k), rng.choice([1, 4, 9], k), rng.integers(50, 401, k)

    abc = []
    for a, g, s in zip(*sizes(case["models"])):
        h = rng.integers(50, s + 1, case["particles"])
        abc.append({"A": int(a), "G": int(g), "S": int(h.max()), "horizons": [int(x) for x in h]})
    mc3 = [{"A": int(a), "G": int(g), "S": int(s)} for a, g, s in zip(*sizes(case["ladders"]))]
    return {"abc": abc, "mc3": mc3, "ladder": 8}


def _requests(case):
    """The burst: models, sample counts, horizons and counterfactuals by the case."""
    return serving.make_requests(case["requests"], rate=1000.0, catalogue_size=len(serving.CATALOGUE),
                                 seed=100 + case["requests"])


def _posterior_draws(spec, centre, rng, n, width=0.1):
    """n parameter vectors around `centre`, inside the (uniform or fixed)
    priors, as a posterior's samples or a set of chains."""
    lo = np.array([p["prior"][1] for p in spec["params"]], dtype=float)
    hi = np.array([p["prior"][2] if p["prior"][0] == "uniform" else p["prior"][1] for p in spec["params"]], dtype=float)
    centre = np.asarray(centre, dtype=float)
    return np.clip(centre + width * (hi - lo) * rng.normal(size=(n, len(lo))), lo, hi)


# ---- what a program has in hand before the call ----

def prepare(case, seed):
    kind = case["kind"]
    rng = np.random.default_rng(seed)
    st = {"case": case, "seed": int(seed)}
    if kind == "batch":
        ub = batch.UnevenBatch(_batch_workload(case), seed=seed)
        st["ub"] = ub
        st["abc_pv"] = specmod.sample_prior(ub.spec0, rng, len(ub.abc_slots))
        st["prop"] = np.clip(ub.pv + rng.normal(0.0, 1.0, ub.pv.shape) * ub.step_sd, ub.lo, ub.hi)
        return st
    if kind == "weights":
        n, v = case["particles"], case["variables"]
        sd = rng.uniform(0.1, 2.0, v)
        mix = rng.normal(0, 1, (v, v)) / math.sqrt(v) * 0.5 + np.eye(v)
        st["prev"] = rng.uniform(1, 5, v) + rng.normal(0, 1, (n, v)) @ mix * sd
        w = rng.gamma(2.0, 0.5, n)
        st["w"] = w / w.mean()
        cov = np.cov(st["prev"].T).reshape(v, v)
        st["inv_M"] = np.linalg.inv(cov)
        st["size"] = 0.5
        pick = rng.choice(n, n, p=w / w.sum())
        st["theta"] = st["prev"][pick] + st["size"] * rng.multivariate_normal(np.zeros(v), cov, n)
        st["logprior"] = rng.normal(-3.0, 0.5, n)
        return st
    if kind == "serving":
        st["server"] = serving.PredictionServer(serving.CATALOGUE, t_post=100, max_horizon=180,
                                                nposterior=case["posterior"], hbm_budget=24 << 30, max_pool=1000,
                                                chunk=14, seed=seed % 1000003)
        return st
    if kind == "load":
        spec, truth = _model("spatial", case["areas"], 4, case["days"])
        n = case["n"]
        st["pv"] = _posterior_draws(spec, truth, rng, n)
        st["counts"] = [_replay(spec, _tables(spec, pv), rng=rng)["counts"] for pv in st["pv"]]
        st["ctx"] = _lib.Context(spec, capacity=n, nslot=n)
        return st
    spec, truth = _case_model(case)
    n = case["n"]
    st["key"] = rng.integers(0, 1 << 31, n, dtype=np.int64).astype(np.uint32)
    st["inst"] = np.arange(n, dtype=np.int32)
    if kind == "filter":
        st["ctx"] = _lib.Context(spec, capacity=n, nslot=1)
        st["pv"] = _posterior_draws(spec, truth, rng, 1, width=0.01)
        return st
    if kind == "proposals":
        ctx = st["ctx"] = _lib.Context(spec, capacity=2 * n, nslot=2 * n)
        cur = _posterior_draws(spec, truth, rng, n)
        st["prop_pv"] = _posterior_draws(spec, cur, rng, n, width=0.02)
        st["prop"] = st["inst"] + n
        st["Pr"], _ = ctx.set_param(st["inst"], cur)
        ctx.simulate(st["inst"], st["inst"], st["key"], seed=seed, stream=1)
        ctx.obs_loglik(st["inst"])
        st["mask"] = None
        if case["mask"]:
            st["mask"] = (rng.random((n, case["days"], case["areas"])) < case["mask"]).astype(np.uint8)
        return st
    ctx = st["ctx"] = _lib.Context(spec, capacity=n, nslot=n)
    st["pv"] = specmod.sample_prior(spec, rng, n)
    if kind == "tables":
        ctx.set_param(st["inst"], st["pv"])
        ctx.simulate(st["inst"], st["inst"], st["key"], seed=seed, stream=1)
    return st


# ---- one pass ----

def run(st):
    case, seed = st["case"], st["seed"]
    return _RUN[case["kind"]](st, case, seed)


def _run_generation(st, case, seed):
    """Fresh parameters, simulation, log-likelihood; a single particle's
    program also reads its trajectory."""
    ctx, inst = st["ctx"], st["inst"]
    prior, inside = ctx.set_param(inst, st["pv"])
    ctx.simulate(inst, inst, st["key"], seed=seed, stream=2)
    out = {"prior": prior, "inside": inside, "loglik": ctx.obs_loglik(inst)}
    if case["n"] == 1:
        out["transnum"] = ctx.get_transnum(0)
    return out


def _run_proposals(st, case, seed):
    ctx, inst, prop = st["ctx"], st["inst"], st["prop"]
    prior, _ = ctx.set_param(prop, st["prop_pv"])
    ctx.mbp(inst, prop, prop, st["key"], simu_mask=st["mask"], seed=seed, stream=3)
    loglik = ctx.obs_loglik(prop)
    al, accepted = ctx.accept(inst, prop, 1, prior - st["Pr"], st["key"], invT=0.1, seed=seed, stream=3)
    return {"prior": prior, "loglik": loglik, "al": al, "accepted": accepted}


def _run_batch(st, case, seed):
    """The work of batch.UnevenBatch.sweep for given proposals."""
    ub = st["ub"]
    h = np.concatenate([ub.h_abc, ub.h_mc3])
    slots = np.concatenate([ub.abc_slots, ub.alt.reshape(-1)])
    prior, _ = _lib.batch_set_param(h, slots, np.concatenate([st["abc_pv"], st["prop"].reshape(-1, ub.nparam)]))
    rec, na = ub.sweep_records()
    _stats, loglik = _lib.run_batch(rec, seed=seed, stream=100, loglik=True)
    ratio = prior[na:] - ub.Pr.reshape(-1)
    al, accepted = _lib.batch_accept(rec[na:], ub.invT_chains, ratio, mode=1, seed=seed, stream=100)
    order, ntr, nac = _lib.batch_mc3_swap_arrays(ub.ladder_ptr, ub.h_mc3, ub.cur.reshape(-1), 0, ub.invT_chains,
                                                 seed=seed, stream=100)
    return {"prior": prior, "loglik": loglik, "al": al, "accepted": accepted, "order": order, "trials": ntr, "swaps": nac}


def _run_filter(st, case, seed):
    """A PMCMC proposal: parameters, likelihood estimate, the sampled
    trajectory's infections."""
    ctx, inst = st["ctx"], st["inst"]
    ctx.set_param([0], st["pv"])
    estimate, ancestors = ctx.pmcmc_obs_prob(inst, 0, st["key"], invT=1.0, seed=seed, stream=4)
    ctx.pmcmc_particle_sample(0)
    tr = 1 if case["model"] == "dense" else 0
    return {"estimate": estimate, "ancestors": ancestors, "infections": ctx.sum_transnum([0], tr, 0, ctx.S)}


def _run_tables(st, case, seed):
    loglik, errors = st["ctx"].obs_loglik(st["inst"], with_dt=True)
    return {"loglik": loglik, "errors": errors}


def _run_load(st, case, seed):
    ctx, n = st["ctx"], case["n"]
    inst = np.arange(n, dtype=np.int32)
    prior, _ = ctx.set_param(inst, st["pv"])
    for k in range(n):
        ctx.put_transnum(k, k, st["counts"][k])
    loglik, errors = ctx.obs_loglik(inst, with_dt=True)
    return {"prior": prior, "loglik": loglik, "errors": errors, "state_loglik": ctx.pois_loglik(inst),
            "means": np.stack([ctx.get_transmean(k) for k in range(n)]),
            "pops": np.stack([ctx.get_pop(k) for k in range(n)])}


def _run_weights(st, case, seed):
    return _lib.abcsmc_weights(st["prev"], st["w"], st["theta"], st["inv_M"], st["size"], st["logprior"])


def _run_serving(st, case, seed):
    requests = _requests(case)
    return [r.result for r in st["server"].run(requests, realtime=False)]


_RUN = {"generation": _run_generation, "proposals": _run_proposals, "batch": _run_batch, "filter": _run_filter,
        "tables": _run_tables, "load": _run_load, "weights": _run_weights, "serving": _run_serving}


# ---- what a pass cannot do without ----

def _step_work(A, G, C, T, nnz):
    """Operations of one instance's step: per transition a mean, a quarter of a
    10-round generator block and a short inversion; per cell the age mixing;
    per mixing entry and group a multiply-add."""
    AG = A * G
    return AG * (T * (4 + 15 + 20) + 2 * G) + 2 * nnz * G


def _nnz(spec):
    return len(spec["M"]["to"]) if spec.get("M") is not None else 0


def _sim_work(spec, n, steps, words):
    """n instances over `steps` steps, `words` 4-byte trajectory values kept
    per cell and step, plus the final populations and the slot tables."""
    A, G, C, T, S = _dims(spec)
    AG = A * G
    return n * (4 * AG * (steps * words + C) + 12 * steps), n * steps * _step_work(A, G, C, T, _nnz(spec))


def _obs_work(spec, n, counts_only=False):
    """The likelihood: an int32 count per element, per observation its value
    and two constants (shared by the instances)."""
    if spec.get("obs_table") is not None:
        nobs, nel = len(spec["obs_table"]["y"]), len(spec["obs_table"]["y"]) * len(spec["obs_table"]["dp"])
    else:
        nobs = len(spec["obs"])
        nel = sum((o["sett_f"] - o["sett_i"]) * len(o["area"]) * len(o["dp"]) * len(o["tr"]) for o in spec["obs"])
    return 4 * nel * n + 24 * nobs + 8 * n, n * (nel + 5 * nobs)


def work(case):
    kind = case["kind"]
    if kind == "weights":
        n, v = case["particles"], case["variables"]
        return {"bytes": 8 * (2 * n * v + 3 * n + v * v), "flops": n * n * (2 * v + 30)}
    if kind == "serving":
        b = f = 0
        for r in _requests(case):
            A, G = serving.CATALOGUE[r.model]
            b += r.nsamp * 4 * A * G * (r.horizon * 3 + 8)
            f += r.nsamp * r.horizon * _step_work(A, G, 4, 3, A * min(10, A - 1))
        return {"bytes": b, "flops": f}
    if kind == "batch":
        b = f = 0
        wl = _batch_workload(case)
        for g in wl["abc"]:
            AG, steps = g["A"] * g["G"], sum(g["horizons"])
            b += 4 * AG * 3 * steps + 4 * g["A"] * g["G"] * steps
            f += steps * _step_work(g["A"], g["G"], 4, 3, 10 * g["A"])
        for m in wl["mc3"]:
            AG, steps = m["A"] * m["G"], 8 * m["S"]
            b += 4 * AG * 12 * steps + 4 * AG * steps
            f += steps * _step_work(m["A"], m["G"], 4, 3, 10 * m["A"])
        return {"bytes": b, "flops": f}
    if kind == "load":
        spec, _ = _model("spatial", case["areas"], 4, case["days"])
        A, G, C, T, S = _dims(spec)
        n = case["n"]
        return {"bytes": n * 4 * A * G * S * (2 * T + C), "flops": n * S * A * G * (T * 30 + 2 * G) + _obs_work(spec, n)[1]}
    if kind == "filter":
        # The model's observations come of a simulation; their sizes are known without it.
        A, G, days, n = case["areas"], case["groups"], case["days"], case["n"]
        C, T = (10, 11) if case["model"] == "dense" else (4, 3)
        nnz = A * (A - 1) if case["model"] == "dense" else A * min(10, A - 1)
        return {"bytes": n * 4 * A * G * days * (2 * T + C + 1), "flops": n * days * _step_work(A, G, C, T, nnz)}
    spec, _ = _case_model(case)
    A, G, C, T, S = _dims(spec)
    n = case["n"]
    ob, of = _obs_work(spec, n)
    if kind == "tables":
        return {"bytes": ob, "flops": of}
    sb, sf = _sim_work(spec, n, S, 2 * T + C)
    if kind == "proposals":
        sb += n * 8 * A * G * T * S                            # the current chains' counts and means
    return {"bytes": sb + ob, "flops": sf + of}


# ---- the same in 64 bits, by plain numpy ----

def _log_prior(spec, pv):
    """The log prior density: uniform and fixed priors only."""
    total = sum(-math.log(p["prior"][2] - p["prior"][1]) for p in spec["params"] if p["prior"][0] == "uniform")
    return np.full(len(pv), total)


def _tables(spec, pv):
    """Rates, infectivities, beta(t), contact matrix and area mixing of the
    spatial model for one parameter vector."""
    A, G, C, T, S = _dims(spec)
    pv = np.array(pv, dtype=np.float64)
    for d in spec.get("dirichlet", []):
        pv[d["param"]] = pv[d["param"]] / pv[d["param"]].sum()
    pop = np.asarray(spec["pop"], dtype=np.float64)            # [A][C][G]
    area_pop, group_pop, total = pop.sum((1, 2)), pop.sum((0, 1)), pop.sum()
    N = np.asarray(spec["N"], dtype=np.float64) / (group_pop[:, None] / total)
    N = 0.5 * (N + N.T)
    N /= (group_pop @ N).sum() / (G * total)
    mix = np.zeros((A, A))
    for c in range(A):
        a, b = spec["M"]["rowptr"][c], spec["M"]["rowptr"][c + 1]
        mix[c, spec["M"]["to"][a:b]] += spec["M"]["val"][a:b]
        mix[c, c] += spec["M"]["diag"][c]
    mix /= (mix @ area_pop)[:, None]
    nexit = np.bincount([t["from"] for t in spec["trans"]], minlength=C)
    rate, inf = np.zeros(T), np.array([pv[c["inf"]] if c["inf"] >= 0 else 0.0 for c in spec["comps"]])
    for k, t in enumerate(spec["trans"]):
        if not t.get("infection"):
            rate[k] = 1.0 / pv[spec["comps"][t["from"]]["mean"][0]]
            if nexit[t["from"]] > 1:
                rate[k] *= pv[t["prob"][0]]
    # Expected infectivity x time of one infection, over the transition graph
    # (rates do not depend on the group), times the contact matrix' growth.
    itr = [k for k, t in enumerate(spec["trans"]) if t.get("infection")][0]
    V = np.eye(C) * 1e-300
    for k, t in enumerate(spec["trans"]):
        if k != itr:
            V[t["from"], t["from"]] += rate[k]
            V[t["to"], t["from"]] -= rate[k]
    live = [c for c in range(C) if V[c, c] > 1e-200]
    occupancy = np.linalg.solve(V[np.ix_(live, live)], np.eye(len(live))[:, live.index(spec["trans"][itr]["to"])])
    growth = np.abs(np.linalg.eigvals((group_pop / total)[:, None] * N)).max()
    ratio = float(occupancy @ inf[live]) * growth
    spl = spec["splines"][spec["R_spline"]]
    R = np.interp((np.arange(S) + 0.5) * spec["period"] / S, spl["t"], pv[spl["param"]])
    return {"rate": rate, "inf": inf, "beta": R / ratio, "N": N, "mix": mix, "itr": itr}


def _replay(spec, tb, counts=None, rng=None):
    """Means and populations of a trajectory in 64 bits: of given counts, or
    of counts drawn step by step, as a saved posterior sample holds them."""
    A, G, C, T, S = _dims(spec)
    pop = np.asarray(spec["pop"], dtype=np.float64)
    out = {"means": np.zeros((S, A, T, G)), "pops": np.zeros((S, A, C, G)),
           "counts": np.zeros((S, A, T, G), dtype=np.int32) if counts is None else counts}
    for s in range(S):
        out["pops"][s] = pop
        force = tb["beta"][s] * np.maximum((tb["mix"].T @ np.einsum("acg,c->ag", pop, tb["inf"])) @ tb["N"].T, 0.0)
        nxt = pop.copy()
        for k, t in enumerate(spec["trans"]):
            src = np.maximum(pop[:, t["from"]], 0.0)
            m = out["means"][s, :, k] = src * (force if k == tb["itr"] else tb["rate"][k])
            if counts is None:
                out["counts"][s, :, k] = np.minimum(rng.poisson(m), np.maximum(nxt[:, t["from"]], 0.0))
            nxt[:, t["from"]] -= out["counts"][s, :, k]
            nxt[:, t["to"]] += out["counts"][s, :, k]
        pop = nxt
    return out


def _exact_load(case, seed):
    spec, truth = _model("spatial", case["areas"], 4, case["days"])
    rng = np.random.default_rng(seed)
    pvs = _posterior_draws(spec, truth, rng, case["n"])
    counts = [_replay(spec, _tables(spec, pv), rng=rng)["counts"] for pv in pvs]
    y = np.array([o["y"] for o in spec["obs"]])
    graph, table = np.array([o["graph"] for o in spec["obs"]]), np.array([o["datatable"] for o in spec["obs"]])
    day, area = np.array([o["sett_i"] for o in spec["obs"]]), np.array([o["area"][0] for o in spec["obs"]])
    tr = np.array([o["tr"][0] for o in spec["obs"]])
    top = np.zeros(graph.max() + 1)
    np.maximum.at(top, graph, y)
    sd = (0.99 * y + 0.01 * top[graph]) * 0.1
    out = {"loglik": [], "errors": [], "state_loglik": [], "means": [], "pops": None}
    lgam = np.cumsum(np.concatenate([[0.0], np.log(np.arange(1, 1 + max(int(c.max()) for c in counts) + 1))]))
    for pv, cnt in zip(pvs, counts):
        r = _replay(spec, _tables(spec, pv), counts=cnt)
        v = cnt.sum(-1, dtype=np.float64)[day, area, tr]
        term = -0.5 * np.log(2 * np.pi * sd * sd) - (y - v) ** 2 / (2 * sd * sd)
        out["loglik"].append(math.fsum(term))
        out["errors"].append([-2 * math.fsum(term[table == d]) for d in range(table.max() + 1)])
        lam = r["means"]
        with np.errstate(divide="ignore", invalid="ignore"):
            lp = np.where(lam == 0, np.where(cnt == 0, 0.0, -1e9), np.where(cnt == 0, -lam, cnt * np.log(lam) - lam - lgam[cnt]))
        out["state_loglik"].append(math.fsum(lp.reshape(-1)))
        out["means"].append(lam)
    return {"prior": _log_prior(spec, pvs), "loglik": np.array(out["loglik"]), "errors": np.array(out["errors"]),
            "state_loglik": np.array(out["state_loglik"]), "means": np.stack(out["means"]), "pops": None}


def exact(case, seed):
    """Where an output is a function of the inputs that plain numpy gives:
    densities, importance weights and everything computed from loaded samples.
    What follows from the framework's own random draws has no such value."""
    kind = case["kind"]
    if kind == "weights":
        st = prepare(case, seed)
        out = np.empty(len(st["theta"]))
        for i, th in enumerate(st["theta"]):
            e = (th - st["prev"]) / st["size"]
            out[i] = math.exp(st["logprior"][i]) / (st["w"] @ np.exp(-0.5 * ((e @ st["inv_M"]) * e).sum(1)))
        return out
    if kind == "load":
        return _exact_load(case, seed)
    if kind == "generation":
        spec, _ = _case_model(case)
        return {"prior": _log_prior(spec, np.zeros(case["n"])), "inside": None, "loglik": None}
    return None
