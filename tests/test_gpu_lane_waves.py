"""Waves that give an env A lanes beside and instead of waves of 64 envs: batches past the
small ones all at once and in rounds, and hybrid workgroups of table waves and one to three
LDS waves.  At batch sizes that leave the last wave and the last ticket part-filled, on maps
whose codes end inside a word, against the oracle bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

STATE = ("s", "ep_step", "episode", "reward", "done", "action")


def check(gpu, oracle, N, W, H, A, chunks, resident=0, variant=0, hybrid=False, cells=0, block=None, kernel=None, **kw):
    cr = None
    if cells:
        cls, start, cr = gpu.gen_maps_noise(3, N, W, H, 4, 0.2, 0.3, 5.0)
    else:
        cls, start = gpu.gen_maps_bernoulli(7, N, N, W, H, 0.12, 0.08)
    cfg = gpu.make_config(N, W, H, n_actions=A, reward_flags=cells, lr=0.3, gamma=0.9, seed=N + A, trap_reward=-0.5,
                          **{"eps0": 0.4, "episode_len": 9, **kw})
    with gpu.Engine(cfg, 0) as eng:
        eng.set_maps(cls, start, cr)
        eng.set_resident_envs(resident)
        eng.set_fused_variant(variant)
        for c in chunks:
            plan = eng.fused_kernel_info(c)
            assert ("hbm+lds" in plan["name"]) == hybrid, plan
            assert hybrid or kernel or plan["name"] == "k_fused_lanes<%d,fast%s>" % (A, ",cells" if cells else ""), plan
            assert kernel is None or plan["name"] == kernel, plan
            assert block is None or plan["block"] == block, plan
            eng.run_fused(c)
            assert sum(eng.fused_split()) == N
        q, st = eng.q_get(0, N), eng.get_state()
        stats = eng.episode_stats() if cfg.track_returns else None
    Q = np.zeros((N, W * H, A), np.float32)
    ost = oracle.new_state(cfg, start)
    ostats = oracle.new_stats(N) if cfg.track_returns else None
    oracle.run(cfg, cls, cr, start, Q, ost, 0, sum(chunks), stats=ostats)
    for k in STATE:
        assert np.array_equal(st[k], ost[k]), k
    assert np.array_equal(q.reshape(Q.shape), Q)
    for k in stats or ():
        assert np.array_equal(stats[k], ostats[k]), k


# one wave to a workgroup; `resident`: in rounds drawn from the counter (from 64 steps on) or
# dealt by position
@pytest.mark.parametrize("N,W,H,A,chunks,resident,kw", [
    (16387, 13, 11, 4, (8, 9, 64), 0, dict()),
    (16385, 9, 7, 8, (8, 31), 0, dict(eps_mode=3, eps0=1.0, eps_end=0.1, eps_span=4, max_mode=1)),
    (33001, 5, 3, 4, (65, 20), 3000, dict()),
    (33001, 5, 3, 8, (65, 20), 3000, dict(track_returns=1, max_episodes=3)),
    (20003, 7, 5, 4, (130, 12), 4096, dict(cells=1, eps_mode=3, eps0=0.9, eps_end=0.2, eps_span=5)),
    (20003, 7, 5, 8, (130, 12), 0, dict(cells=3, max_mode=1)),
    (99001, 9, 7, 4, (70,), 0, dict(max_mode=1)),  # more than the registers hold at once: two even rounds
])
def test_lane_waves(gpu, oracle, N, W, H, A, chunks, resident, kw):
    check(gpu, oracle, N, W, H, A, chunks, resident, block=64, **kw)


# table waves and LDS waves: three, two and one of them, fewer envs than a wave, than a round
@pytest.mark.parametrize("N,W,H,A,lds_waves", [(4099, 6, 5, 4, 3), (4099, 6, 5, 8, 3), (2051, 16, 16, 4, 2), (1033, 16, 16, 8, 2),
                                               (1037, 20, 19, 4, 1), (521, 23, 21, 8, 1), (1, 16, 16, 4, 2), (7, 3, 3, 8, 3)])
def test_hybrid_workgroups(gpu, oracle, N, W, H, A, lds_waves):
    check(gpu, oracle, N, W, H, A, (67, 130, 1), variant=2, hybrid=True, block=64 * (2 + lds_waves))


# waves of 64 envs, which short calls of more envs than lane waves are for take, and longer calls on
# tables past the caches (which keep rows in LDS: with staged move codes below); the general loop's
# hybrid workgroups
LINEAR = dict(eps_mode=3, eps0=0.9, eps_end=0.1, eps_span=4)


@pytest.mark.parametrize("N,W,H,A,chunks,variant,kernel,kw", [
    (17003, 13, 11, 4, (3, 1, 7), 0, "k_fused_tickets<4,fast,hbm>", dict()),
    (17003, 13, 11, 8, (3, 1, 7), 0, "k_fused_tickets<8,fast,hbm>", dict()),
    (17003, 13, 11, 4, (3, 1, 7), 0, "k_fused_tickets<4,fast+,hbm>", LINEAR),
    (17003, 13, 11, 8, (3, 1, 7), 0, "k_fused_tickets<8,fast+,hbm>", dict(cells=3)),
    (65601, 32, 31, 4, (130, 2), 0, "k_fused_tickets<4,fast,hbm>", dict()),
    (70003, 16, 16, 8, (130, 2), 1, "k_fused_tickets<8,fast,hbm>", dict()),
    (65601, 32, 31, 4, (130, 2), 0, "k_fused_tickets<4,fast+,hbm>", LINEAR),
    (70003, 16, 16, 8, (130, 2), 0, "k_fused_tickets<8,fast+,hbm>", LINEAR),
    (4099, 6, 5, 4, (67, 30), 2, "k_fused_tickets<4,general,hbm+lds>", dict(goal_mode=1)),
    (4099, 6, 5, 8, (67, 30), 2, "k_fused_tickets<8,general,hbm+lds>", dict(goal_mode=1)),
])
def test_waves_of_64_envs(gpu, oracle, N, W, H, A, chunks, variant, kernel, kw):
    check(gpu, oracle, N, W, H, A, chunks, variant=variant, hybrid="hbm+lds" in kernel, kernel=kernel, **kw)


# those that keep no rows in LDS: class maps staged, move codes staged (from 128 steps on)
@pytest.mark.parametrize("N,W,H,A,steps,codes,kw", [
    (17003, 31, 33, 4, 7, 0, dict()), (34001, 20, 20, 4, 5, 0, LINEAR), (34001, 20, 20, 8, 5, 0, dict()), (17003, 31, 33, 8, 7, 0, dict(cells=3)),
    (48001, 29, 29, 4, 131, 1, dict()), (48001, 29, 29, 4, 131, 1, LINEAR), (30001, 24, 24, 8, 131, 1, dict()), (30001, 24, 24, 8, 131, 1, dict(cells=1)),
])
def test_waves_of_64_envs_without_rows(gpu, oracle, N, W, H, A, steps, codes, kw):
    kernel = "k_fused_tickets<%d,fast%s,hbm>" % (A, "+" if kw else "")
    check(gpu, oracle, N, W, H, A, (steps, 1), kernel=kernel, **kw)
    cfg = gpu.make_config(N, W, H, n_actions=A, reward_flags=kw.get("cells", 0), eps_mode=kw.get("eps_mode", 0), eps_span=9)
    assert gpu.fused_plan_rows(cfg, steps) == (0, codes) and gpu.fused_plan_rows(cfg, 1)[0] == 0
