"""An env to as many lanes as it has actions (all tables in LDS, beside their move words or
beside move codes; tables in HBM with codes in LDS or in global memory): every form, at the
batch sizes where envs per wave and waves per workgroup change, with everything an episode's
end can bring along, in launches that begin on odd and even steps and end inside a tape.
Bit for bit against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

STATE = ("s", "ep_step", "episode", "reward", "done", "action")
STATS = ("last_return", "last_length", "return_sum", "length_sum")


def check(gpu, oracle, N, W, H, A, chunks, want_kernel, shared_map=False, cells=0, **kw):
    n_maps = 1 if shared_map else N
    cr = None
    if cells:
        cls, start, cr = gpu.gen_maps_noise(3, n_maps, W, H, 4, 0.2, 0.3, 5.0)
        start = np.resize(start, N).astype(np.int32)
        cls = cls.copy()
        cls[:, 1::7] = np.where(cls[:, 1::7] == 0, 2, cls[:, 1::7])  # traps, which pay by the cell they guard
        cls[np.arange(N) % n_maps, start] = 0
    else:
        cls, start = gpu.gen_maps_bernoulli(7, n_maps, N, W, H, 0.12, 0.08)
    cfg = gpu.make_config(N, W, H, n_actions=A, map_mode=gpu.MAP_SHARED if shared_map else gpu.MAP_PER_ENV,
                          reward_flags=cells, lr=0.3, gamma=0.9, seed=N + A, trap_reward=-0.5,
                          **{"eps0": 0.4, "episode_len": 9, **kw})
    with gpu.Engine(cfg, 0) as eng:
        eng.set_maps(cls, start, cr)
        name = eng.fused_kernel_info(max(chunks))["name"]
        assert name.startswith(want_kernel), name
        for c in chunks:
            eng.run_fused(c)
        q, st = eng.q_get(0, N), eng.get_state()
        stats = eng.episode_stats() if cfg.track_returns else None
    Q = np.zeros((N, W * H, A), np.float32)
    ost = oracle.new_state(cfg, start)
    ostats = oracle.new_stats(N) if cfg.track_returns else None
    oracle.run(cfg, cls, cr, start, Q, ost, 0, sum(chunks), stats=ostats)
    for k in STATE:
        assert np.array_equal(st[k], ost[k]), (k, name)
    assert np.array_equal(q.reshape(Q.shape), Q), name
    if stats:
        for k in STATS:
            assert np.array_equal(stats[k], ostats[k]), (k, name)


@pytest.mark.parametrize("A", [4, 8])
@pytest.mark.parametrize("N", [1, 2, 63, 1023, 1025, 4097, 16385])
def test_tables_in_lds(gpu, oracle, N, A):
    check(gpu, oracle, N, 4, 3, A, (17, 64, 33, 131), "k_fused_tickets_lds<%d,fast>" % A)


@pytest.mark.parametrize("A,N,W,H,shared", [(4, 4, 90, 45, False), (8, 3, 47, 45, False), (4, 1300, 30, 29, False),
                                            (8, 700, 21, 27, True), (4, 1, 80, 81, True), (4, 2050, 25, 23, False)])
def test_tables_in_lds_beside_words_or_codes(gpu, oracle, A, N, W, H, shared):
    check(gpu, oracle, N, W, H, A, (200, 57), "k_fused_per_env_lds" if shared else "k_fused_tickets_lds",
          shared_map=shared, episode_len=60)


@pytest.mark.parametrize("A,N,W,H,shared,cells,kernel", [
    (4, 5000, 24, 21, False, 0, "k_fused_lanes<4,fast>"),      # codes in LDS
    (8, 2049, 24, 21, False, 0, "k_fused_lanes<8,fast>"),
    (4, 700, 9, 7, False, 3, "k_fused_lanes<4,fast,cells>"),        # rewards by cell
    (8, 700, 9, 7, False, 1, "k_fused_lanes<8,fast,cells>"),
    (4, 300, 70, 66, False, 3, "k_fused_per_env<4,2,fast,lanes>"),   # codes in global memory
    (8, 300, 70, 66, False, 1, "k_fused_per_env<8,2,fast,lanes>"),
    (4, 9000, 24, 31, True, 0, "k_fused_per_env<4,1,fast,lanes>"),   # one map's codes in LDS, four waves to a workgroup
    (8, 4000, 24, 31, True, 3, "k_fused_per_env<8,1,fast,lanes>"),
])
def test_tables_in_hbm(gpu, oracle, A, N, W, H, shared, cells, kernel):
    check(gpu, oracle, N, W, H, A, (129, 70, 1), kernel, shared_map=shared, cells=cells, episode_len=40)


@pytest.mark.parametrize("A,N,W,H,shared", [(4, 1, 5, 4, True), (4, 300, 5, 4, True), (8, 77, 5, 4, False),
                                            (4, 3000, 40, 40, True), (4, 6000, 24, 21, False)])
@pytest.mark.parametrize("events", [
    dict(eps_mode=1, eps0=1.0, eps_decay=0.99, eps_span=150),
    dict(eps_mode=2, eps0=1.0, eps_decay=0.8, eps_span=9),
    dict(eps_mode=3, eps0=0.9, eps_end=0.0, eps_span=6, max_mode=1),
    dict(track_returns=1, episode_len=0),
    dict(track_returns=1, max_episodes=5, eps_mode=1, eps_decay=0.999, eps_span=300, max_mode=1),
    dict(track_returns=1, max_episodes=7, eps_mode=3, eps_end=0.1, eps_span=10),
    dict(max_episodes=1),
])
def test_what_an_episodes_end_brings_along(gpu, oracle, A, N, W, H, shared, events):
    check(gpu, oracle, N, W, H, A, (31, 130, 97), "k_fused_", shared_map=shared, **events)
