"""The work that users of this framework have it do, as cases that can be timed.

A case is a dict of plain values; `kind` says which public entry points it goes through:

  env      the drop-in single environment: one gym-shaped step() per pass
  batch    the drop-in Q-learning class: one update_batch() of Python lists, the table read back
  train    the training driver's loop body: one call of `steps` select/step/update rounds with
           episode statistics, then state and statistics read back (as train() does per chunk)
  fused    BatchedEnvironment.run(steps) on envs with a map and a table each
  large    the same on large maps with per-cell rewards and an epsilon that falls by episode
  shared   the same with one map and one table for all envs (ordered sum of the updates)
  rounds   one round of select() / step(actions) / update() / state(), as a caller does who
           looks at every step
  replay   td_update() of a batch of recorded transitions (numpy arrays) on a shared table

All runs start from zero tables (replay: from a filled one), which is where training starts.
The package is taken from the working folder."""
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.getcwd(), "cudarl-arena_amd")
sys.path[:0] = [_PKG, os.path.join(_PKG, "lib")]
import pycrl  # noqa: E402
import cudarl_core  # noqa: E402

LEVELS = 128  # distinct large maps in a level pool; envs share them out


def listed():
    return [
        # the smallest call: a gym loop on the default 10x10 world
        dict(name="env_step", kind="env", width=10, height=10),
        # an agent that learns from small batches through the drop-in class, default table
        dict(name="q_batch", kind="batch", n=256, width=10, height=10, actions=4),
        # the default training run: one env, episodes of at most 500 steps
        dict(name="train_one", kind="train", n=1, width=10, height=10, steps=500),
        # the same training run for a few thousand envs at once
        dict(name="train_4096", kind="train", n=4096, width=10, height=10, steps=500),
        # 4096 independent 32x32 grids, an episode's length per call
        dict(name="fused_4096", kind="fused", n=4096, width=32, height=32, actions=4, steps=256, eps="fixed", floor=False),
        # 1M independent 16x16 grids (4 GB of tables), a whole training run per call
        dict(name="fused_1m", kind="fused", n=1 << 20, width=16, height=16, actions=4, steps=1000, eps="fixed", floor=False),
        # the same in short calls, for a caller that watches the run
        dict(name="fused_1m_short", kind="fused", n=1 << 20, width=16, height=16, actions=4, steps=20, eps="fixed", floor=False),
        # 8192 large grids, 8 actions, cell rewards (16 GB of tables)
        dict(name="large_8192", kind="large", n=8192, width=256, height=256, actions=8, steps=256),
        # 65,536 envs that learn one table together
        dict(name="shared_65536", kind="shared", n=65536, width=64, height=64, actions=4, steps=200),
        # a shared table of a larger, odd-sized map
        dict(name="shared_big_map", kind="shared", n=20000, width=101, height=99, actions=8, steps=50),
        # a caller with its own policy: one round at a time through host arrays
        dict(name="rounds_4096", kind="rounds", n=4096, width=32, height=32, actions=4, shared=False),
        # a replay buffer's worth of transitions on one table
        dict(name="replay_65536", kind="replay", n=65536, width=64, height=64, actions=4),
    ]


def _log(rng, lo, hi):
    return int(round(float(lo) * (float(hi) / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["env", "batch", "train", "fused", "fused", "large", "shared", "rounds", "replay"])
    actions = rng.choice([4, 8])
    if kind == "env":
        return dict(kind=kind, width=rng.randint(5, 64), height=rng.randint(5, 64))
    if kind == "batch":
        return dict(kind=kind, n=_log(rng, 1, 1024), width=rng.randint(5, 24), height=rng.randint(5, 24), actions=actions)
    if kind == "train":
        return dict(kind=kind, n=_log(rng, 1, 16384), width=rng.randint(5, 40), height=rng.randint(5, 40),
                    steps=rng.randint(100, 500))
    if kind == "fused":
        w, h = rng.randint(4, 48), rng.randint(4, 48)
        most = min(1 << 20, (4 << 30) // (w * h * actions * 4))
        return dict(kind=kind, n=_log(rng, 100, most), width=w, height=h, actions=actions, steps=_log(rng, 1, 1000),
                    eps=rng.choice(["fixed", "fixed", "linear"]), floor=rng.random() < 0.2)
    if kind == "large":
        return dict(kind=kind, n=_log(rng, 256, 8192), width=rng.randint(64, 256), height=rng.randint(64, 256),
                    actions=actions, steps=_log(rng, 16, 256))
    if kind == "shared":
        w, h = _log(rng, 8, 128), _log(rng, 8, 128)
        n = _log(rng, 256, 65536)
        # no more than shared_65536 or, for tables past 16,384 entries, shared_big_map
        most = 65536 * 200 // n if w * h * actions <= 16384 else 20000 * 101 * 99 * 8 * 50 // (n * w * h * actions)
        return dict(kind=kind, n=n, width=w, height=h, actions=actions, steps=max(1, min(_log(rng, 1, 256), most)))
    if kind == "rounds":
        return dict(kind=kind, n=_log(rng, 1, 65536), width=rng.randint(8, 40), height=rng.randint(8, 40),
                    actions=actions, shared=rng.random() < 0.4)
    return dict(kind=kind, n=_log(rng, 64, 262144), width=_log(rng, 8, 128), height=_log(rng, 8, 128), actions=actions)


class _DeviceView:
    """A device array of an Engine for torch.as_tensor (no copy)."""

    def __init__(self, engine, which, shape, typestr):
        self.engine = engine
        self.__cuda_array_interface__ = dict(shape=shape, typestr=typestr, data=(engine.device_ptr(which), False),
                                             version=3, strides=None)


_PTR_Q = 6  # include/crl.h, CRL_PTR_Q


def _batched(case, seed, **options):
    """BatchedEnvironment and zero-copy views of everything that a call updates."""
    env = cudarl_core.BatchedEnvironment(n_envs=case["n"], width=case["width"], height=case["height"],
                                         n_actions=case["actions"], seed=seed, **options)
    names = ("s", "ep_step", "episode", "reward", "done", "action", "q")
    return env, {k: torch.utils.dlpack.from_dlpack(env.dlpack(k)) for k in names}


def prepare(case, seed):
    kind, w, h = case["kind"], case["width"], case["height"]
    rng = np.random.RandomState(seed % (1 << 32))
    if kind == "env":
        return dict(kind=kind, env=cudarl_core.PyEnvironment(w, h, seed % (1 << 30)),
                    actions=rng.randint(0, 4, 4096).tolist(), at=0)
    if kind == "batch":
        n = case["n"]
        q = cudarl_core.CudaQLearning(w, h, case["actions"])
        q.set_q_table(rng.uniform(-0.1, 1.0, w * h * case["actions"]).astype(np.float32).tolist())
        x, y = rng.randint(0, w, n), rng.randint(0, h, n)
        x2, y2 = np.clip(x + rng.randint(-1, 2, n), 0, w - 1), np.clip(y + rng.randint(-1, 2, n), 0, h - 1)
        return dict(kind=kind, q=q, s=list(zip(x.tolist(), y.tolist())), s2=list(zip(x2.tolist(), y2.tolist())),
                    a=rng.randint(0, case["actions"], n).tolist(), r=rng.normal(-0.01, 0.1, n).tolist(),
                    done=(rng.rand(n) < 0.02).tolist())
    if kind == "train":
        n = case["n"]
        cfg = pycrl.make_config(n, w, h, map_mode=pycrl.MAP_SHARED, episode_len=case["steps"], lr=0.1, gamma=0.99,
                                eps_mode=pycrl.EPS_STEP_MULT, eps0=1.0, eps_decay=0.995, eps_span=500001,
                                max_episodes=1 << 30, track_returns=1, seed=seed)
        engine = pycrl.Engine(cfg, 0)
        # the default world: everything free, the goal in the top-right corner, starts anywhere else
        cls = np.zeros((1, w * h), np.uint8)
        cls[0, w - 1] = pycrl.CELL_GOAL
        start = rng.randint(0, w * h - 1, n)
        engine.set_maps(cls, (start + (start >= w - 1)).astype(np.int32))
        q = torch.as_tensor(_DeviceView(engine, _PTR_Q, (n, w * h, 4), "<f4"), device="cuda")
        return dict(kind=kind, engine=engine, steps=case["steps"], q=q)
    if kind == "fused":
        eps = dict(exploration_rate=0.1) if case["eps"] == "fixed" else dict(
            exploration_rate=1.0, exploration_end=0.05, eps_span=100, eps_mode=pycrl.EPS_EPISODE_LINEAR)
        env, views = _batched(case, seed, episode_len=128, discount_factor=0.95, max_mode=int(case["floor"]), **eps)
        env.set_maps(*pycrl.gen_maps_bernoulli(seed, case["n"], case["n"], w, h, 0.1, 0.02))
        return dict(kind=kind, env=env, views=views, steps=case["steps"])
    if kind == "large":
        n = case["n"]
        env, views = _batched(case, seed, episode_len=1024, exploration_rate=1.0, exploration_end=0.05, eps_span=100,
                              eps_mode=pycrl.EPS_EPISODE_LINEAR,
                              reward_flags=pycrl.REWARD_CELLS | pycrl.REWARD_BASE_CELLS)
        pool = min(n, LEVELS)
        cls, start, cell_reward = pycrl.gen_maps_noise(seed, pool, w, h)
        at = np.arange(n) % pool
        env.set_maps(cls[at], start[at], cell_reward[at])
        return dict(kind=kind, env=env, views=views, steps=case["steps"])
    # a step size that a table shared by this many envs per cell stays stable with
    n = case["n"]
    lr = min(0.05, 0.008 * w * h / n)
    if kind == "shared":
        env, views = _batched(case, seed, shared_table=True, shared_map=True, learning_rate=lr, exploration_rate=0.2,
                              episode_len=256)
        env.set_maps(*pycrl.gen_maps_bernoulli(seed, 1, n, w, h, 0.15))
        return dict(kind=kind, env=env, views=views, steps=case["steps"])
    if kind == "rounds":
        shared = case["shared"]
        env, views = _batched(case, seed, shared_table=shared, shared_map=shared, exploration_rate=0.2,
                              learning_rate=lr if shared else 0.1, episode_len=128)
        env.set_maps(*pycrl.gen_maps_bernoulli(seed, 1 if shared else n, n, w, h, 0.15))
        return dict(kind=kind, env=env, q=views["q"])
    cfg = pycrl.make_config(1, w, h, n_actions=case["actions"], table_mode=pycrl.TABLE_SHARED,
                            map_mode=pycrl.MAP_SHARED, lr=lr, seed=seed)
    engine = pycrl.Engine(cfg, 0)
    engine.q_set(0, rng.uniform(-0.1, 1.0, w * h * case["actions"]).astype(np.float32))
    x, y = rng.randint(0, w, n), rng.randint(0, h, n)
    x2, y2 = np.clip(x + rng.randint(-1, 2, n), 0, w - 1), np.clip(y + rng.randint(-1, 2, n), 0, h - 1)
    q = torch.as_tensor(_DeviceView(engine, _PTR_Q, (w * h, case["actions"]), "<f4"), device="cuda")
    return dict(kind=kind, engine=engine, q=q, s=(y * w + x).astype(np.int32), s2=(y2 * w + x2).astype(np.int32),
                a=rng.randint(0, case["actions"], n).astype(np.int32), r=rng.normal(-0.01, 0.1, n).astype(np.float32),
                done=(rng.rand(n) < 0.02).astype(np.uint8))


def run(state):
    kind = state["kind"]
    if kind == "env":
        env, at = state["env"], state["at"]
        state["at"] = (at + 1) % 4096
        obs, reward, done, info = env.step(state["actions"][at])
        if done:
            env.reset()
        return obs, reward, done, info["agent_x"], info["agent_y"]
    if kind == "batch":
        q = state["q"]
        q.update_batch(state["s"], state["a"], state["r"], state["s2"], state["done"])
        return np.array(q.get_q_table(), np.float32)
    if kind == "train":
        engine = state["engine"]
        engine.run_fused(state["steps"])
        return engine.get_state(), engine.episode_stats(), state["q"]
    if kind == "rounds":
        env = state["env"]
        actions = env.select()
        env.step(actions)
        env.update()
        return actions, env.state(), state["q"]
    if kind == "replay":
        state["engine"].td_update(0, state["s"], state["a"], state["r"], state["s2"], state["done"])
        return state["q"]
    state["env"].run(state["steps"])
    return state["views"]


def work(case):
    """Each input read once, each output written once; additions, products and comparisons of
    select (A), target and update (A + 4) per env-step or sample."""
    kind, cells = case["kind"], case["width"] * case["height"]
    n, A = case.get("n", 1), case.get("actions", 4)
    row = 4 * A
    steps = case.get("steps", 1)
    state = 4 + 2 * 12 + 6  # start; cell, episode step and episode in and out; reward, done and action out
    flops = n * steps * (2 * A + 4)
    if kind == "env":
        return dict(bytes=4 * cells + 64, flops=16)
    if kind in ("batch", "replay"):  # transitions; the rows they name in and one value out, or the whole table if that is less
        table = min(n * (row + 8), 8 * cells * A) + (4 * cells * A if kind == "batch" else 0)
        return dict(bytes=17 * n + table, flops=n * (A + 6))
    shared = kind == "shared" or case.get("shared", False)
    maps = cells / 4.0 * (1 if shared or kind == "train" else n)  # two bits to a cell
    # a row in and one value out per step, or every table in and out whole if that is less
    tables = min(n * steps * (row + 4), 8 * cells * A * (1 if shared else n))
    extra = 0
    if kind == "train":
        extra = n * 16
    if kind == "large":
        maps = min(maps, n * steps / 4.0)
        extra = n * steps * 4  # a cell's reward per step
    if kind == "rounds":
        maps = min(maps, n * 1.0)
        extra = n * 8  # the actions out and in again
    return dict(bytes=n * state + maps + tables + extra, flops=flops)


def tolerance(case):
    """Every sum has a stated order and every draw a stated stream: results are the same bits
    whatever the launch shape."""
    return "exact"
