"""The one-launch shared-table kernel where each key of the table has its place: threads know the lowest of
their cell before they choose an action.  One cell that all envs stand in (more holders of a key than places to
line up in), the smallest and the largest tables, part-filled blocks, envs whose budget is used up beside others
that go on, calls that begin where others ended.  Bit for bit against the oracle."""
import numpy as np
import pytest

from test_gpu_hashed_tables import run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,W,H,A,kw", [
    (300, 1, 2, 4, dict()), (3001, 2, 2, 8, dict()), (65536, 3, 3, 4, dict()), (257, 64, 64, 4, dict()), (20000, 64, 32, 8, dict()),
    (65536, 64, 64, 4, dict(episode_len=2)), (5000, 7, 5, 8, dict(episode_len=1)),
    (1000, 6, 6, 4, dict(max_episodes=2)), (1000, 8, 9, 8, dict(max_episodes=3, max_mode=1)), (700, 5, 5, 4, dict(auto_reset=0)),
])
@pytest.mark.parametrize("same_start", [True, False])
def test_leads_of_cells(gpu, oracle, N, W, H, A, kw, same_start):
    cls, start = gpu.gen_maps_bernoulli(3, 1, N, W, H, 0.1 if W * H > 8 else 0.0, 0.0)
    if same_start:
        start[:] = start[0]
    options = dict(episode_len=9)
    options.update(kw)
    cfg = gpu.make_config(N, W, H, n_actions=A, table_mode=gpu.TABLE_SHARED, map_mode=gpu.MAP_SHARED,
                          lr=min(0.02, 0.005 * W * H / N), eps0=0.5, seed=17, **options)
    name, q = run(gpu, oracle, cfg, cls, start, (17, 16, 20))
    plain = set(kw) <= {"episode_len"}
    assert name == "k_shared_persist<%d,1%s>" % (A, ",folded" if plain else "") and np.count_nonzero(q) > 0
