"""What a user of this framework has it do, as cases that can be timed and compared: environment pools stepped by a
random policy, a training loop's batched environments, flat expansions, breadth-first searches and the state set, through
the public entry points of mymyr_amd. `listed` names the cases, `draw` gives more of the same ranges, `prepare` makes
what a program has in hand before a call (on the GPU), `run` is one call or one turn of the program's loop.

Every result is whole numbers (state words, counts, ids, flags) or rewards that are sums of two constants, so results are
compared exactly."""

from __future__ import annotations

import os
import random

import numpy as np
import torch

from mymyr_amd import batched, gen, hip, rl, search, workloads
from mymyr_amd.task import Task

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
TASKS = os.path.join(ROOT, "tests", "golden", "tasks")


def listed() -> list[dict]:
    return [
        # the gridworld workload: few envs, where one step is launch and latency (a small agent's rollout loop)
        {"name": "pool_gridworld_1k", "kind": "pool", "domain": "gridworld", "width": 32, "height": 32, "envs": 1024, "encode": 0, "warm": 24},
        # the transport workload: an ordinary rollout batch over a lifted, typed domain
        {"name": "pool_transport_64k", "kind": "pool", "domain": "transport", "locations": 64, "trucks": 16, "packages": 128,
         "envs": 65536, "encode": 0, "warm": 12},
        # the transport_xl workload: the largest batch, with the true-atom index tensor and the masks that a learner reads
        {"name": "pool_transport_xl_256k", "kind": "pool", "domain": "transport", "locations": 128, "trucks": 32, "packages": 512,
         "envs": 262144, "encode": 544, "warm": 4},
        # a trainer's loop over a table of instances of several sizes: actions chosen outside, final states kept, visited
        # tables, truncation and autoreset into sampled instances, an odd number of envs
        {"name": "batched_table_20k", "kind": "batched", "locations": 24, "trucks": 6, "packages": 40, "instances": 3, "envs": 20011,
         "max_steps": 24, "warm": 8},
        # one planner decision: the successors of a few states with their hashes and goal flags
        {"name": "expand_transport_64", "kind": "expand", "locations": 24, "trucks": 6, "packages": 40, "rows": 64, "k": 64},
        # every successor of a batch of states, flat and as the padded view that a learner scores
        {"name": "expand_transport_8k", "kind": "expand", "locations": 64, "trucks": 16, "packages": 128, "rows": 8195, "k": 256},
        # a short plan: the shortest path in the gridworld, many small layers
        {"name": "brfs_gridworld_goal", "kind": "brfs_grid", "width": 32, "height": 32},
        # a benchmark domain explored to its end (376,832 states over ground actions)
        {"name": "brfs_gripper_all", "kind": "brfs_file", "file": "gripper__prob05", "max_states": 0},
        # a lifted task with wide rows (176 words) searched to a budget of a million states
        {"name": "brfs_transport_1m", "kind": "brfs_transport", "locations": 64, "trucks": 16, "packages": 128, "max_states": 1000000},
        # the strips workload, the headline: a frontier that explodes, stopped by its budget
        {"name": "brfs_strips_64m", "kind": "brfs_strips", "props": 512, "actions": 4096, "max_states": 1 << 26},
        # the dedup workload at a quarter of its rows: rows with 30% duplicates in batches of 2^20
        {"name": "dedup_16m", "kind": "dedup", "rows": 1 << 24, "words": 16, "batch": 1 << 20},
        # the public hash of an odd number of rows of an odd width
        {"name": "hash_rows_1m", "kind": "hash", "rows": 1000003, "words": 13},
    ]


def _log_int(rng: random.Random, lo: int, hi: int) -> int:
    """A whole number of [lo, hi], even over its logarithm."""
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng: random.Random) -> dict:
    kind = rng.choice(["pool_grid", "pool_transport", "batched", "expand", "brfs_grid", "brfs_transport", "brfs_strips", "dedup", "hash"])
    if kind == "pool_grid":
        return {"kind": "pool", "domain": "gridworld", "width": rng.randint(5, 36), "height": rng.randint(5, 36),
                "envs": _log_int(rng, 1, 65536), "encode": rng.choice([0, 1]), "warm": rng.randint(1, 24)}
    if kind == "pool_transport":
        # up to the largest listed step's words and envs
        trucks, packages = _log_int(rng, 2, 32), _log_int(rng, 3, 512)
        locations = rng.randint(6, 128)
        words = (trucks + packages) * locations // 64 + trucks * packages // 64 + 1
        envs = _log_int(rng, 1, min(262144, (1344 * 262144) // (2 * words)))
        return {"kind": "pool", "domain": "transport", "locations": locations, "trucks": trucks, "packages": packages, "envs": envs,
                "encode": rng.choice([0, trucks + packages]), "warm": rng.randint(1, 6)}
    if kind == "batched":
        return {"kind": "batched", "locations": rng.randint(6, 64), "trucks": rng.randint(2, 16), "packages": _log_int(rng, 3, 128),
                "instances": rng.randint(1, 4), "envs": _log_int(rng, 1, 32768), "max_steps": rng.randint(8, 48), "warm": rng.randint(1, 10)}
    if kind == "expand":
        locations, trucks, packages = rng.randint(6, 64), rng.randint(2, 16), _log_int(rng, 3, 128)
        return {"kind": "expand", "locations": locations, "trucks": trucks, "packages": packages, "rows": _log_int(rng, 1, 8192),
                "k": rng.choice([16, 64, 100, 256])}
    if kind == "brfs_grid":
        return {"kind": "brfs_grid", "width": rng.randint(8, 32), "height": rng.randint(8, 32)}
    if kind == "brfs_transport":
        return {"kind": "brfs_transport", "locations": rng.randint(6, 64), "trucks": rng.randint(2, 16), "packages": _log_int(rng, 3, 128),
                "max_states": _log_int(rng, 1000, 1000000)}
    if kind == "brfs_strips":
        return {"kind": "brfs_strips", "props": rng.randint(100, 512), "actions": _log_int(rng, 300, 4096),
                "max_states": _log_int(rng, 4096, 1 << 25)}
    if kind == "dedup":
        words = rng.randint(1, 40)
        return {"kind": "dedup", "rows": _log_int(rng, 1000, (1 << 28) // max(words, 16)), "words": words, "batch": 1 << rng.randint(14, 20)}
    return {"kind": "hash", "rows": _log_int(rng, 100, 1000000), "words": _log_int(rng, 1, 200)}


def _transport(case: dict, k: int = 0) -> Task:
    """The k-th transport instance of a case: the first as stated, the next ones a quarter smaller each."""
    cut = lambda v, least: max(least, v * (4 - k) // 4)  # noqa: E731
    return Task.from_text(gen.transport(cut(case["locations"], 6), cut(case["trucks"], 1), cut(case["packages"], 2),
                                        goals=min(32, cut(case["packages"], 2)), seed=k))


def _pool_task(case: dict) -> Task:
    if case["domain"] == "gridworld":
        return Task.from_text(gen.gridworld(case["width"], case["height"], 0.2, seed=0))
    return _transport(case)


def _walked(task: Task, rows: int, seed: int, steps: int = 6) -> torch.Tensor:
    """States of random walks from the initial state ([rows, words] on the GPU), as a program has them in hand."""
    pool = rl.DeviceEnvPool(task, rows, seed=seed, max_steps=None)
    pool.reset()
    for _ in range(steps):
        pool.step()
    return pool.states.clone()


def _host_row(states: torch.Tensor) -> np.ndarray:
    return states[0].cpu().numpy().view(np.uint64).copy()


def prepare(case: dict, seed: int) -> dict:
    kind = case["kind"]
    st = {"case": case}
    if kind == "pool":
        # a pool some steps into its episodes (the policy's random key is the seed)
        task = _pool_task(case)
        pool = rl.DeviceEnvPool(task, case["envs"], seed=seed, step_reward=-1.0, goal_reward=1.0)
        pool.reset()
        for _ in range(case["warm"]):
            pool.step(encode=case["encode"], labels=False)
        st.update(task=task, pool=pool)
    elif kind == "batched":
        tasks = [_transport(case, k) for k in range(case["instances"])]
        env = batched.BatchedEnv(tasks if len(tasks) > 1 else tasks[0], case["envs"], seed=seed, max_steps=case["max_steps"],
                                 step_reward=-1.0, goals=True, track_visited=True)
        for _ in range(case["warm"]):
            env.step(None, final=False, copy=False)
        st.update(tasks=tasks, env=env)
    elif kind == "expand":
        task = _transport(case)
        st.update(task=task, states=_walked(task, case["rows"], seed))
    elif kind == "brfs_grid":
        task = Task.from_text(gen.gridworld(case["width"], case["height"], 0.2, seed=0))
        st.update(task=task, start=_host_row(_walked(task, 1, seed, 8)), options={})
    elif kind == "brfs_file":
        task = Task.from_text_file(os.path.join(TASKS, case["file"] + ".txt"))
        st.update(task=task, start=_host_row(_walked(task, 1, seed)), options={"stop_at_goal": False})
    elif kind == "brfs_transport":
        task = _transport(case)
        st.update(task=task, start=_host_row(_walked(task, 1, seed)), options={"max_states": case["max_states"]})
    elif kind == "brfs_strips":
        # start states as the workload's own: an eighth of the propositions, drawn at random
        task = Task.from_text(gen.random_strips(case["props"], case["actions"], init_atoms=case["props"] // 8, seed=workloads.SEED), "dense")
        rng = random.Random(seed)
        start = np.zeros(task.words, np.uint64)
        for p in rng.sample(range(case["props"]), case["props"] // 8):
            start[p // 64] |= np.uint64(1 << (p % 64))
        st.update(task=task, start=start, options={"max_depth": workloads.STRIPS.max_depth, "max_states": case["max_states"], "stop_at_goal": False})
    elif kind == "dedup":
        st.update(rows=hip.dedup_rows(0, case["rows"], case["words"], seed=seed, dup=workloads.DEDUP_DUP),
                  set=hip.StateSet(case["rows"], case["words"], 0.5, batch=case["batch"]))
    elif kind == "hash":
        g = torch.Generator(device="cuda").manual_seed(seed)
        rows = torch.randint(-2**62, 2**62, (case["rows"], case["words"]), dtype=torch.int64, device="cuda", generator=g)
        rows[:: 7, case["words"] - 1] = 0  # rows whose trailing words are zero hash shorter
        st.update(rows=rows)
    return st


def run(state: dict):
    case = state["case"]
    kind = case["kind"]
    if kind == "pool":
        r = state["pool"].step(encode=case["encode"], labels=False)
        return {k: r[k] for k in ("states", "reward", "terminated", "truncated", "count", "steps", "at_goal", "goal", "atoms", "masks") if k in r}
    if kind == "batched":
        # the policy acts on the counts of its observation; here it takes the random policy's choice
        env = state["env"]
        r = env.step(env.random_actions())
        return {"reward": r.reward, "terminated": r.terminated, "truncated": r.truncated, "goal": r.goal, "invalid": r.invalid,
                "schema": r.schema, "binding": r.binding, "final_states": r.final_states, "count": r.count, "states": r.states,
                "task_ids": r.task_ids, "at_goal": r.at_goal, "revisited": r.revisited}
    if kind == "expand":
        # the flat arrays' lengths follow the states, so the padded view (every successor up to k of a state) is returned
        x = rl.expand(state["task"], state["states"], goal=True, hashes=True)
        p = rl.pad(x, case["k"])
        return {"offsets": x["offsets"], "generated": x["generated"], "total": x["total"],
                **{k: p[k] for k in ("index", "mask", "count", "succ", "schema", "binding", "goal", "succ_hash")}}
    if kind in ("brfs_grid", "brfs_file", "brfs_transport", "brfs_strips"):
        r = search.brfs(state["task"], start=state["start"], fingerprint=True, **state["options"])
        layers = np.full((1024, 3), -1, np.int64)
        plan = np.full((1024, 8), -1, np.int64)
        for i, row in enumerate(r.layer_counts[:1024]):
            layers[i] = row
        for i, a in enumerate(r.plan[:1024]):
            plan[i, : 1 + len(a.binding)] = (a.schema, *a.binding)
        return {"states": r.states, "expanded": r.expanded, "generated": r.generated, "goals": r.num_goal_states, "layers": r.layers,
                "fingerprint": np.array([r.fingerprint], np.uint64).view(np.int64), "layer_counts": layers, "plan": plan, "cost": r.cost}
    if kind == "dedup":
        s, rows, batch = state["set"], state["rows"], case["batch"]
        s.clear()
        new = [s.insert(rows[b: b + batch], want_ids=False, count=False)[2] for b in range(0, case["rows"], batch)]
        return {"unique": len(s), "is_new": torch.cat(new)}
    return {"hash": hip.hash_rows(state["rows"])}


def _words(case: dict) -> int:
    """State words of a case's (first) task, as its dense or reachable layout has them."""
    if case.get("domain") == "gridworld" or case["kind"] == "brfs_grid":
        return max(1, int(case["width"] * case["height"] * 0.8 + 63) // 64)
    L, T, P = case["locations"], case["trucks"], case["packages"]
    return ((T + P) * L + T * P + 63) // 64


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind == "pool":
        # the row read and the words of a move's two effects written, the row's scalars in and out, and the encoding
        per = 8 * _words(case) + 16 + 8 * 4 + 30 + (4 * case["encode"] + 3 if case["encode"] else 0)
        return {"bytes": float(case["envs"] * per), "flops": 0.0}
    if kind == "batched":
        # besides: the final states written, the observation's copies of states and goal masks
        return {"bytes": float(case["envs"] * (8 * _words(case) * 8 + 100)), "flops": 0.0}
    if kind == "expand":
        # about two loads or unloads per three packages and the roads out of the trucks' locations
        succ = case["packages"] * case["trucks"] // max(1, case["locations"]) + case["trucks"] * 4 + 1
        R = 8 * _words(case)
        # the flat successors written and the padded view of them
        return {"bytes": float(case["rows"] * (R + (succ + case["k"]) * (R + 8 + 4 + 4 + 12 + 1))), "flops": 0.0}
    if kind == "brfs_grid":
        return {"bytes": float(0.8 * case["width"] * case["height"] * (16 * _words(case) + 16)), "flops": 0.0}
    if kind == "brfs_file":
        # 376,832 states of one word, 2,031,616 successors: each state stored and read, a table entry per successor probed
        return {"bytes": float(376832 * 32 + 2031616 * 8), "flops": 0.0}
    if kind == "brfs_transport":
        return {"bytes": float(case["max_states"] * (8 * _words(case) + 24)), "flops": 0.0}
    if kind == "brfs_strips":
        # a new state stored (row, table entry, node), about three more successors per new state that are duplicates
        W = (case["props"] + 63) // 64
        return {"bytes": float(case["max_states"] * (8 * W + 16 + 3 * 8)), "flops": 0.0}
    if kind == "dedup":
        # every row read once, a table entry each, the new rows (seven in ten) written once
        R = 8 * case["words"]
        return {"bytes": float(case["rows"] * (R + 8 + 1 + 0.7 * R)), "flops": 0.0}
    return {"bytes": float(case["rows"] * (8 * case["words"] + 8)), "flops": 0.0}


def tolerance(case: dict):
    return "exact"


def exact(case: dict, seed: int):
    """Whole numbers have no rounding to measure; the cases' results are compared bit for bit."""
    return None
