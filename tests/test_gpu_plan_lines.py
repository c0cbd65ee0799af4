"""Both sides of the lines where a fused launch changes its kernel: tables in LDS or behind lane
waves, lane waves in rounds dealt or drawn, hybrid workgroups or rounds of lane waves, waves of 64
envs that keep rows in LDS or none.  Against the oracle bit for bit."""
import numpy as np
import pytest

from test_gpu_lane_waves import STATE, check

pytestmark = pytest.mark.gpu

LDS, LANES, PLAIN, HYBRID = "k_fused_tickets_lds<%d,fast>", "k_fused_lanes<%d,fast>", "k_fused_tickets<%d,fast,hbm>", "k_fused_tickets<%d,fast,hbm+lds>"
ROWS = PLAIN + ", rows kept"  # which go by the name of the plain ones


@pytest.mark.parametrize("N,W,H,A,steps,kernel", [
    (2046, 15, 17, 4, 16, LDS),                                      # 8 KB to a wave: from the first
    (4090, 16, 16, 4, 39, LANES), (4090, 16, 16, 4, 40, LDS),        # 16 KB to a wave
    (15001, 8, 8, 4, 40, LDS), (30001, 8, 8, 4, 117, LANES), (30001, 8, 8, 4, 119, LDS),  # four and eight such waves
    (70, 47, 49, 8, 143, LANES), (70, 47, 49, 8, 144, LDS),          # 72 KB to a wave
    (33001, 32, 32, 4, 130, PLAIN), (33001, 32, 32, 4, 25, ROWS), (33001, 32, 32, 4, 26, PLAIN),  # a map costs more to stage
    (40001, 8, 8, 4, 7, PLAIN), (62001, 16, 16, 4, 2, PLAIN), (62001, 16, 16, 4, 3, ROWS),  # few envs; a part-filled last wave
    (50001, 32, 32, 4, 63, ROWS), (50001, 32, 32, 4, 64, LANES),     # rounds, of at most 65,536 envs
    (66001, 28, 28, 4, 130, ROWS), (66001, 28, 28, 4, 131, LANES),   # of more
    (250001, 8, 8, 4, 9, ROWS), (250001, 8, 8, 4, 10, LANES),        # in place of hybrid workgroups
    (250001, 8, 8, 4, 71, LANES), (250001, 8, 8, 4, 72, HYBRID),
    (94001, 12, 12, 4, 47, ROWS), (94001, 12, 12, 4, 48, LANES),     # ... where they are few rounds
    (200001, 8, 8, 4, 5, ROWS), (200001, 8, 8, 4, 6, ROWS),
])
def test_lines(gpu, oracle, N, W, H, A, steps, kernel):
    cls, start = gpu.gen_maps_bernoulli(7, N, N, W, H, 0.12, 0.08)
    cfg = gpu.make_config(N, W, H, n_actions=A, lr=0.3, gamma=0.9, seed=N + A, eps0=0.4, episode_len=9)
    Q, want = np.zeros((N, W * H, A), np.float32), oracle.new_state(cfg, start)
    oracle.run(cfg, cls, None, start, Q, want, 0, steps)
    with gpu.Engine(cfg, 0) as eng:
        eng.set_maps(cls, start)
        kept = gpu.fused_plan_rows(cfg, steps)[0] != 0
        assert eng.fused_kernel_info(steps)["name"] + (", rows kept" if kept else "") == kernel % A
        eng.run_fused(steps)
        state = eng.get_state()
        assert all(np.array_equal(state[k], want[k]) for k in STATE)
        assert np.array_equal(eng.q_get(0, N).reshape(Q.shape), Q)


# rounds of lane waves, dealt by position and drawn from the counter (from 256 steps on, with 8
# actions or more than three rounds); the last one partly filled
@pytest.mark.parametrize("N,W,H,A,resident,steps", [
    (5003, 5, 3, 4, 1600, 255), (5003, 5, 3, 4, 1600, 256), (5003, 5, 3, 4, 1700, 257), (17003, 5, 3, 4, 1600, 256),
    (5003, 5, 3, 8, 4000, 255), (5003, 5, 3, 8, 4000, 256), (5003, 5, 3, 8, 500, 300),
])
def test_rounds_of_lane_waves(gpu, oracle, N, W, H, A, resident, steps):
    check(gpu, oracle, N, W, H, A, (steps, 9, steps), resident, kernel="k_fused_lanes<%d,fast>" % A)


@pytest.mark.parametrize("N,W,H,A,steps", [(50001, 40, 40, 4, 64)])
def test_uneven_rounds_of_lane_waves(gpu, oracle, N, W, H, A, steps):
    """Six waves of 26,704 bytes of LDS to a compute unit where even rounds would need seven: they draw their envs."""
    with gpu.Engine(gpu.make_config(N, W, H, n_actions=A, max_mode=gpu.MAX_ZERO_FLOOR), 0) as eng:
        assert eng.fused_kernel_info(steps)["grid"] == 1536
    check(gpu, oracle, N, W, H, A, (steps,), kernel="k_fused_lanes<%d,fast>" % A, max_mode=gpu.MAX_ZERO_FLOOR)


def test_tables_read_ahead(gpu):
    """Seven rounds of lane waves on tables past the caches: read ahead whole from 160 steps on, not in shorter calls."""
    N, W, A = 147500, 16, 8
    cls, start = gpu.gen_maps_bernoulli(7, N, N, W, W, 0.1, 0.02)
    cfg = gpu.make_config(N, W, W, n_actions=A, episode_len=40, eps0=0.2, seed=3)
    with gpu.Engine(cfg, 0) as one, gpu.Engine(cfg, 0) as two:
        for e in (one, two):
            e.set_maps(cls, start)
            assert e.fused_kernel_info(160)["name"] == "k_fused_lanes<8,fast>"
        for _ in range(2):
            one.run_fused(160)
            two.run_fused(159)
            two.run_fused(1)
        a, b = one.get_state(), two.get_state()
        assert all(np.array_equal(a[k], b[k]) for k in STATE)
        for at in range(0, N, 29500):
            assert np.array_equal(one.q_get(at, 29500), two.q_get(at, 29500))


@pytest.mark.parametrize("N,W,H,A", [(98500, 16, 16, 4), (74000, 12, 16, 8)])
def test_tables_read_ahead_in_four_rounds(gpu, N, W, H, A):
    """Four rounds of lane waves, epsilon by episode: tables read ahead from 200 steps on, not in shorter calls."""
    cls, start = gpu.gen_maps_bernoulli(7, N, N, W, H, 0.1, 0.02)
    cfg = gpu.make_config(N, W, H, n_actions=A, episode_len=40, eps0=0.9, eps_mode=gpu.EPS_EPISODE_LINEAR, eps_end=0.1,
                          eps_span=9, seed=3)
    with gpu.Engine(cfg, 0) as one, gpu.Engine(cfg, 0) as two:
        for e in (one, two):
            e.set_maps(cls, start)
        plan = one.fused_kernel_info(200)
        assert plan["name"] == "k_fused_lanes<%d,fast>" % A
        waves = -(-N // (64 // A))
        assert 3 * plan["grid"] < waves <= 4 * plan["grid"]
        for _ in range(2):
            one.run_fused(200)
            two.run_fused(199)
            two.run_fused(1)
        a, b = one.get_state(), two.get_state()
        assert all(np.array_equal(a[k], b[k]) for k in STATE)
        for at in range(0, N, N // 2):
            assert np.array_equal(one.q_get(at, N // 2), two.q_get(at, N // 2))
