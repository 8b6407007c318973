"""What a user of the plan evaluator has it do, as cases that can be timed: single evaluations through the calls that
carry the reference's names, the handful of candidates of a search step, host and device batches of the five
workloads of `rpeg_amd.configs` from a few hundred plans to their full candidate sets, a whole search, and a
population of annealing chains.

A case is a dict of plain values with a `kind`:

  evaluate   evaluate_cached(configuration, cache, ...) for one plan after another: what a pipeline calls for its start
             plans and its results, schedule included
  map        evaluate_batch([configurations]): the candidates of a search step, as objects of the plan representation
  mass       Engine.eval_mass(batch): host tensors, critical-chain masses too (a step of an annealing loop)
  util       Engine.eval_util(batch): host tensors, utilisation too (a window of polish() under that objective)
  host       Engine.eval(batch): host tensors in, host arrays out
  device     Engine.eval_device(batch): tensors that stay on the device, a population scored in place
  search     search_plan(...): start plans, optimize() over the structural families, polish()
  chains     optimize_chains(...): a population of annealing chains

`workload` is a configuration of `rpeg_amd.configs`: 1 PPO on 32 devices (7B models), 2 GRPO on 128, 3 PPO with and
without actor-critic sharing on 256 (13B), 4 DPO on 1,024 (70B, most plans do not fit), 5 PPO on 512 (70B actor).

A program keeps one engine per problem and hands it batch after batch; so do these cases, and so do the drop-in calls
by themselves.
"""

import dataclasses
import math

import numpy as np

from rpeg_amd import configs
from rpeg_amd.engine.runtime import DeviceBatch, Engine
from rpeg_amd.search import candidates
from rpeg_amd.search.cache import EvalCache
from rpeg_amd.search.evaluate import Configuration, evaluate_batch, evaluate_cached
from rpeg_amd.search.moves import build_candidate_directory, directory_arrays
from rpeg_amd.search.optimizer import OptimizerConfig, optimize_chains, plan_row
from rpeg_amd.search.pipeline import search_plan

ALGORITHM = {1: "ppo", 2: "grpo", 3: "ppo", 4: "dpo", 5: "ppo"}
# per plan: int16 fields of the vertices and four header bytes in, three doubles and a mask byte out
PLAN_BYTES = {1: 149, 2: 109, 3: 149, 4: 89, 5: 149}
# per plan: additions, multiplications, divisions and comparisons in fp64 of cost model, memory model and scheduler,
# averaged over the seeded candidate sets
PLAN_FLOPS = {1: 3697.0, 2: 2165.3, 3: 6502.9, 4: 1245.8, 5: 4155.6}
NODES = {1: 110, 2: 70, 3: 190, 4: 30, 5: 120}   # lowered nodes of a typical plan
# largest device batch drawn: the candidate set of the workload, and the size of config 2's where that is small
MOST = {1: 65536, 2: 131072, 3: 262144, 4: 1048576, 5: 131072}


def listed():
    return [
        # one plan at a time: what the reference's evaluate_cached serves, and what a user tries first
        dict(name="evaluate_ppo", kind="evaluate", workload=1, n=1),
        # K_x = 6 candidates of one iteration of optimize(), as configuration objects
        dict(name="map_ppo_6", kind="map", workload=5, n=6),
        # the proposals of one step of a third of 64 chains
        dict(name="mass_ppo_100", kind="mass", workload=5, n=100),
        # a vertex window of polish() when utilisation is part of the objective
        dict(name="util_acshare_41", kind="util", workload=3, n=41),
        # a caller without device tensors: an odd number of plans, staged through the library
        dict(name="host_grpo_9001", kind="host", workload=2, n=9001),
        # the candidate sets of the workloads, resident on the device
        dict(name="device_ppo_4096", kind="device", workload=1, n=4096),
        dict(name="device_ppo_20011", kind="device", workload=5, n=20011),
        dict(name="device_grpo_65536", kind="device", workload=2, n=65536),
        dict(name="device_acshare_262144", kind="device", workload=3, n=262144),
        dict(name="device_dpo_1048576", kind="device", workload=4, n=1048576),
        # the whole search of the pipeline, on a budget of 1,200 evaluations
        dict(name="search_ppo", kind="search", workload=1, e_max=1200, e_struct=200),
        # the annealing workload: 64 chains of 2,000 steps, six candidates each
        dict(name="chains_64x2000", kind="chains", workload=5, chains=64, steps=2000),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["evaluate", "map", "mass", "util", "host", "host", "device", "device", "device", "device",
                       "search", "chains"])
    w = rng.choice([1, 2, 3, 4, 5])
    if kind == "evaluate":
        return dict(kind=kind, workload=w, n=_log_int(rng, 2, 24))
    if kind == "map":
        return dict(kind=kind, workload=w, n=_log_int(rng, 1, 64))
    if kind == "mass":
        return dict(kind=kind, workload=w, n=_log_int(rng, 1, 1500))
    if kind == "util":
        return dict(kind=kind, workload=w, n=_log_int(rng, 1, 300))
    if kind == "host":
        return dict(kind=kind, workload=w, n=_log_int(rng, 200, 131072))
    if kind == "device":
        return dict(kind=kind, workload=w, n=_log_int(rng, 500, MOST[w]))
    if kind == "search":
        return dict(kind=kind, workload=w, e_max=_log_int(rng, 100, 1200), e_struct=_log_int(rng, 50, 250))
    chains = _log_int(rng, 8, 128)
    return dict(kind="chains", workload=rng.choice([1, 2, 5]), chains=chains,
                steps=_log_int(rng, 50, min(2000, 128000 // chains)))


# ----------------------------------------------------------------------------- preparation
_ENGINES = {}      # one engine per workload for the life of the program
_DIRECTORIES = {}  # and the candidate directory of its template


def _engine(w):
    if w not in _ENGINES:
        _ENGINES[w] = Engine(configs.config(w).problem, "cuda:0")
    return _ENGINES[w]


def _directory(w):
    if w not in _DIRECTORIES:
        p = configs.config(w).problem
        rpeg = p.template(0, ())
        table, _ = build_candidate_directory(rpeg, p.suite, p.device_space, p.workload, _engine(w))
        _DIRECTORIES[w] = directory_arrays(rpeg, table)
    return _DIRECTORIES[w]


def _configurations(cfg, n, seed, tag):
    """n seeded plans of the workload's first template, in the plan representation."""
    p = dataclasses.replace(cfg.problem, structures=cfg.problem.structures[:1])
    batch = candidates.generate(p, n, cfg.tau_choices, seed=seed, tag=tag)
    out = []
    for i in range(n):
        rpeg, plan, _ = batch.configuration(p, i)
        out.append(Configuration(rpeg, plan, p.device_space))
    return out


def prepare(case, seed):
    w, kind = case["workload"], case["kind"]
    cfg = configs.config(w)
    p = cfg.problem
    state = dict(kind=kind, problem=p)
    if kind in ("evaluate", "map"):
        state["configs"] = _configurations(cfg, case["n"], seed, w)
    elif kind in ("mass", "util", "host", "device"):
        state["engine"] = _engine(w)
        batch = candidates.generate(p, case["n"], cfg.tau_choices, seed=seed, tag=w)
        if kind == "device":
            state["batch"] = DeviceBatch(batch, "cuda:0")
            state["out"] = state["engine"].alloc_outputs(batch.n)
        else:
            state["batch"] = batch
    elif kind == "search":
        state.update(seed=seed, algorithm=ALGORITHM[w],
                     opt=OptimizerConfig(E_max=case["e_max"], E_struct=case["e_struct"], algorithm=ALGORITHM[w]))
    else:
        state.update(seed=seed, engine=_engine(w), directory=_directory(w), chains=case["chains"], steps=case["steps"],
                     variants=[(0, 0), (1, 0)] if ALGORITHM[w] == "ppo" else [(0,), (1,)],
                     opt=OptimizerConfig(K_x=6, T_init=0.05, T_min=0.05, T_warm=0.10, stag_window=10))
    return state


# ----------------------------------------------------------------------------- one pass
def run(state):
    p, kind = state["problem"], state["kind"]
    if kind == "device":
        return state["engine"].eval_device(state["batch"], state["out"])
    if kind == "host":
        return state["engine"].eval(state["batch"])
    if kind == "mass":
        return state["engine"].eval_mass(state["batch"])
    if kind == "util":
        return state["engine"].eval_util(state["batch"])
    if kind == "evaluate":
        cache = EvalCache()
        got = [evaluate_cached(c, cache, p.suite, p.workload, p.hw, p.K_eval) for c in state["configs"]]
        times = np.zeros((len(got), 2, 512))     # start and finish of the plan's nodes in dispatch order (at most 384 here)
        for g, t in zip(got, times):
            t[0, :len(g[1].start)] = list(g[1].start.values())
            t[1, :len(g[1].finish)] = list(g[1].finish.values())
        return dict(score=np.array([g[0] for g in got]), feasible=np.array([g[2] for g in got]), times=times)
    if kind == "map":
        r = evaluate_batch(state["configs"], p.suite, p.workload, p.hw, p.K_eval)
        return dict(score=r.score, makespan=r.makespan, peak=r.peak, mask=r.mask, feasible=r.feasible)
    if kind == "search":
        r = search_plan(p.suite, p.workload, p.hw, p.device_space, p.K_eval, state["opt"], algorithm=state["algorithm"],
                        seed=state["seed"])
        return dict(start=plan_row(r.start.rpeg, r.start.plan), optimized=plan_row(r.optimized.rpeg, r.optimized.plan),
                    polished=plan_row(r.polished.rpeg, r.polished.plan), scores=r.scores, evaluated=r.cache.size())
    r = optimize_chains(p, state["opt"], state["chains"], state["steps"], state["variants"], seed=state["seed"],
                        engine=state["engine"], directory=state["directory"])
    return dict(best_plan=r.best_plan, best_score=r.best_score, best_step=r.best_step, best_feasible=r.best_feasible,
                cur_plan=r.cur_plan, cur_score=r.cur_score, restarts=r.restarts, n_eval=r.n_eval, dead=r.dead, log=r.log)


def work(case):
    """Plan fields in and results out, each once, and the arithmetic of the plans evaluated."""
    w, kind = case["workload"], case["kind"]
    if kind == "search":
        plans = case["e_max"] + 200          # the budget, the start plans and the windows of polish()
    elif kind == "chains":
        plans = int(4.5 * case["chains"] * case["steps"])   # candidates left after the moves that find none
    else:
        plans = case["n"]
    more = {"mass": 48, "util": 8, "chains": 48, "search": 48, "evaluate": 16 * NODES[w]}.get(kind, 0)
    return {"bytes": plans * (PLAN_BYTES[w] + more), "flops": plans * PLAN_FLOPS[w]}


def tolerance(case):
    """Every double is the one the reference's float64 expressions give, in their order: the same bits."""
    return "exact"
