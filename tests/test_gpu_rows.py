"""64-env waves that keep the rows their envs come to in LDS: maps in LDS or move codes that come with
the rows, four places for them or six, runs cut off at the map's edge, episodes that end at the goal or by the clock in every
other step (the run that leaves may be the one just updated), part-filled last waves, launches that
begin on odd steps.  Bit for bit against the oracle."""
import pytest

from test_gpu_lane_waves import LINEAR, check

pytestmark = pytest.mark.gpu

PLACE = 64 * 32  # bytes: 32 for each of 64 envs


def rows_check(gpu, oracle, N, W, H, A, chunks, staged, places=lambda steps: 4, **kw):
    cfg = gpu.make_config(N, W, H, n_actions=A, reward_flags=kw.get("cells", 0), episode_len=kw.get("episode_len", 9),
                          **{k: v for k, v in kw.items() if k.startswith("eps") or k == "max_mode"})
    for c in chunks:
        plan = gpu.fused_plan_for_config(cfg, c)
        assert plan["lds_bytes"] == places(c) * (PLACE + 64 * (2 if staged else 4)) + (W * H + 15) // 16 * 256 * staged, plan
        assert (plan["grid"], plan["block"]) == (-(-N // 64), 64), plan
        assert gpu.fused_plan_rows(cfg, c)[0] == places(c), plan
    rich = kw.get("cells") or "eps_mode" in kw
    check(gpu, oracle, N, W, H, A, chunks, kernel="k_fused_tickets<%d,fast%s,hbm>" % (A, "+" if rich else ""), **kw)


@pytest.mark.parametrize("kw", [dict(), LINEAR, dict(cells=1), dict(cells=3, **LINEAR), dict(episode_len=1), dict(episode_len=2),
                                dict(episode_len=0)])
@pytest.mark.parametrize("N,W,H,A", [(65603, 13, 11, 4), (65601, 16, 21, 4), (65537, 9, 10, 8)])
def test_short_calls(gpu, oracle, N, W, H, A, kw):
    rows_check(gpu, oracle, N, W, H, A, (1, 7, 2, 5, 7, 7, 7), True, **kw)


@pytest.mark.parametrize("N,W,H,A,steps,kw", [
    (262144, 5, 3, 4, 55, dict()), (262145, 4, 4, 8, 72, dict()), (262207, 1, 7, 4, 33, dict()), (262147, 2, 2, 8, 40, dict(episode_len=2)),
    (262147, 7, 2, 4, 47, dict(max_mode=1)), (262147, 3, 3, 8, 150, dict(max_mode=1, **LINEAR)),
    (262147, 6, 5, 4, 80, dict(cells=3, episode_len=3)), (262147, 3, 6, 8, 50, dict(cells=1, max_mode=1)),
    (98305, 5, 4, 4, 88, dict()), (200000, 3, 3, 8, 50, dict()), (200001, 9, 8, 4, 90, dict()), (82500, 13, 13, 4, 40, dict(episode_len=30)),
    (131073, 5, 5, 4, 60, LINEAR), (98309, 9, 8, 4, 140, dict(max_mode=1)), (82501, 13, 13, 4, 101, dict(max_mode=1, **LINEAR)),
    (262147, 5, 5, 4, 40, dict(LINEAR, episode_len=1)), (262149, 4, 5, 4, 60, dict(episode_len=5)), (262149, 3, 7, 8, 110, dict(episode_len=40)),
])
def test_many_envs(gpu, oracle, N, W, H, A, steps, kw):
    rows_check(gpu, oracle, N, W, H, A, (steps, 9, 31), True, lambda c: 6 if c >= 32 and not ("eps_mode" in kw or "cells" in kw) else 4, **kw)


@pytest.mark.parametrize("N,W,H,A,chunks,kw", [
    (50003, 33, 31, 4, (63, 12), dict()), (65701, 31, 33, 4, (101, 12), LINEAR), (17003, 35, 33, 8, (12, 11, 12), dict()),
    (17003, 34, 34, 8, (12, 14, 11), dict(cells=3, **LINEAR)), (33001, 33, 31, 4, (25, 11), dict()), (16449, 61, 45, 4, (33, 20), LINEAR),
])
def test_codes_with_the_rows(gpu, oracle, N, W, H, A, chunks, kw):
    rows_check(gpu, oracle, N, W, H, A, chunks, False, episode_len=17, **kw)


@pytest.mark.parametrize("N,W,H,A,steps", [(66001, 27, 29, 4, 99), (66001, 27, 29, 4, 100), (66001, 31, 24, 8, 130)])
def test_six_places_on_larger_maps(gpu, oracle, N, W, H, A, steps):
    rows_check(gpu, oracle, N, W, H, A, (steps,), True, lambda c: 6 if c >= 100 else 4, episode_len=30)
