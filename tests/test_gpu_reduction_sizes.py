"""The ordered sum of an update at the sizes where it changes its form: one workgroup of one,
two and four blocks, two launches with one and more groups and more groups than an owner has
waves, tables with a part of a row to an owner up to more owners than compute units, blocks
that hold more keys of one owner than a cell takes.  Bit for bit against the oracle: every sum
has a stated order."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def transitions(rng, S, A, n, cells=None):
    s = rng.choice(cells, n) if cells is not None else rng.integers(0, S, n)
    r = (rng.normal(0, 1, n) * 10.0 ** rng.integers(-3, 3, n)).astype(np.float32)
    a = rng.integers(0, A, n)
    a[rng.random(n) < 0.02] = -1
    return s, a, r, rng.integers(0, S, n), (rng.random(n) < 0.2).astype(np.uint8)


def check(gpu, oracle, W, H, A, batches, mode=0):
    S = W * H
    cfg = gpu.make_config(1, W, H, n_actions=A, max_mode=mode, table_mode=gpu.TABLE_SHARED, map_mode=gpu.MAP_SHARED)
    want = np.random.default_rng(S).normal(0, 1, S * A).astype(np.float32)
    with gpu.Engine(cfg, 0) as eng:
        eng.q_set(0, want)
        for b in batches:
            eng.td_update(0, *b)
            oracle.td_update_batch(want, S, A, *b, 0.1, 0.99, mode)
        assert np.array_equal(eng.q_get(0).reshape(-1), want)


@pytest.mark.parametrize("n", [1, 255, 256, 257, 512, 513, 1023, 1024, 1025, 4096, 4097, 65536, 65537, 70000])
@pytest.mark.parametrize("W,H,A", [(3, 3, 4), (64, 64, 4), (101, 99, 8)])
def test_sample_counts(gpu, oracle, n, W, H, A):
    rng = np.random.default_rng(n)
    # (several calls without a wait between: their pages are taken in turn)
    check(gpu, oracle, W, H, A, [transitions(rng, W * H, A, n) for _ in range(6)], mode=n & 1)


PIECE = 1 << 18  # transitions of a call that go through one page


@pytest.mark.parametrize("n", [PIECE - 1, PIECE, PIECE + 1, 2 * PIECE + 257, 5 * PIECE - 300])
@pytest.mark.parametrize("W,H,A", [(8, 8, 4), (101, 99, 8), (1025, 1024, 4)])  # 1.05 million cells: the scan
def test_batches_of_several_pieces(gpu, oracle, n, W, H, A):
    """Calls large and small in turn, so that pages of one call's pieces are another's."""
    if W > 1000 and n > PIECE + 1:
        n = 2 * PIECE + 1
    rng = np.random.default_rng(n)
    big = transitions(rng, W * H, A, n)
    check(gpu, oracle, W, H, A, [big, transitions(rng, W * H, A, 5000), transitions(rng, W * H, A, 700), big])


@pytest.mark.parametrize("N,W,H,A", [((1 << 21) + 300, 8, 8, 4),   # 2.1 million samples
                                     ((1 << 23) + 300, 16, 16, 4),  # 256 owners' cells outgrow their limit: 16 owners
                                     (140000, 1024, 1024, 4)])      # 4096 owners
def test_very_large_batches_take_two_passes(gpu, oracle, N, W, H, A):
    cls, start = gpu.gen_maps_bernoulli(2, 1, N, W, H, 0.15)
    cfg = gpu.make_config(N, W, H, n_actions=A, table_mode=gpu.TABLE_SHARED, map_mode=gpu.MAP_SHARED, lr=1e-6, eps0=0.3,
                          episode_len=2, seed=6)
    with gpu.Engine(cfg, 0) as eng:
        eng.set_maps(cls, start)
        assert eng.fused_kernel_info(3)["name"] == "k_shared_act+k_reduce_owners"
        eng.run_fused(3)
        q, st = eng.q_get(0), eng.get_state()
    Q = np.zeros((1, W * H, A), np.float32)
    ost = oracle.new_state(cfg, start)
    oracle.run(cfg, cls, None, start, Q, ost, 0, 3)
    assert np.array_equal(q, Q[0]) and np.array_equal(st["s"], ost["s"])


def test_a_late_piece_that_is_refused_leaves_the_table_alone(gpu, oracle):
    W, H, A = 12, 10, 4
    S, n = W * H, 3 * PIECE
    rng = np.random.default_rng(3)
    good = transitions(rng, S, A, n)
    cfg = gpu.make_config(1, W, H, table_mode=gpu.TABLE_SHARED, map_mode=gpu.MAP_SHARED)
    want = rng.normal(0, 1, S * A).astype(np.float32)
    with gpu.Engine(cfg, 0) as eng:
        eng.q_set(0, want)
        for at, which in ((n - 1, 0), (PIECE + 5, 3), (0, 0)):
            bad = [x.copy() for x in good]
            bad[which][at] = S if which else -1
            with pytest.raises(gpu.CrlError, match=r"\[%d\]" % at):
                eng.td_update(0, *bad)
            assert np.array_equal(eng.q_get(0).reshape(-1), want)
        eng.td_update(0, *good)
        oracle.td_update_batch(want, S, A, *good, 0.1, 0.99, 0)
        assert np.array_equal(eng.q_get(0).reshape(-1), want)


@pytest.mark.parametrize("W,H,A", [(16, 16, 8), (16, 17, 8), (64, 65, 4), (181, 181, 8), (400, 400, 8)])
def test_table_sizes(gpu, oracle, W, H, A):
    rng = np.random.default_rng(W)
    check(gpu, oracle, W, H, A, [transitions(rng, W * H, A, 9000)])


@pytest.mark.parametrize("W,H,A", [(64, 64, 4), (101, 99, 8)])
@pytest.mark.parametrize("n", [900, 9000])
def test_crowded_keys_and_cells_that_overflow(gpu, oracle, W, H, A, n):
    S = W * H
    rng = np.random.default_rng(n)
    # whole rows of one owner: cell = (hi << 8) | ((owner - 37 hi) & 255)
    rows = np.array([c for c in ((h << 8) | ((5 - 37 * h) & 255) for h in range(S >> 8)) if c < S])
    check(gpu, oracle, W, H, A, [transitions(rng, S, A, n, rows), transitions(rng, S, A, n, np.array([7])),
                                 transitions(rng, S, A, n, rng.integers(0, S, 12))])


@pytest.mark.parametrize("n", [1, 256, 300, 1024])
def test_collected_changes_are_the_table(gpu, oracle, n):
    W, H, A = 12, 11, 8
    S = W * H
    rng = np.random.default_rng(n)
    b = transitions(rng, S, A, n)
    cfg = gpu.make_config(1, W, H, n_actions=A, table_mode=gpu.TABLE_SHARED, map_mode=gpu.MAP_SHARED)
    mine = rng.normal(0, 1, S * A).astype(np.float32)
    with gpu.Engine(cfg, 0) as eng:
        eng.q_set(0, mine)
        keys, values = eng.td_update_collect(0, *b)
        got = eng.q_get(0).reshape(-1)
        with pytest.raises(gpu.CrlError):
            eng.td_update_collect(0, *transitions(rng, S, A, 1025))
    named = keys[keys >= 0]
    assert len(set(named.tolist())) == len(named)
    assert set(named.tolist()) == set((b[0] * A + b[1])[b[1] >= 0].tolist())
    mine[named] = values[keys >= 0]
    assert np.array_equal(mine, got)


def test_update_of_a_shared_table_from_the_last_step(gpu, oracle):
    for N in (1, 300, 1024, 1025, 5000):
        W, H = 90, 70  # 25,200 keys
        cls, start = gpu.gen_maps_bernoulli(2, 1, N, W, H, 0.15)
        cfg = gpu.make_config(N, W, H, table_mode=gpu.TABLE_SHARED, map_mode=gpu.MAP_SHARED, lr=0.02, eps0=0.3,
                              episode_len=5, seed=3)
        with gpu.Engine(cfg, 0) as eng:
            eng.set_maps(cls, start)
            for _ in range(9):
                eng.select(fetch=False)
                eng.step()
                eng.update()
            q, st = eng.q_get(0), eng.get_state()
        Q = np.zeros((1, W * H, 4), np.float32)
        ost = oracle.new_state(cfg, start)
        oracle.run(cfg, cls, None, start, Q, ost, 0, 9)
        assert np.array_equal(q, Q[0]) and np.array_equal(st["s"], ost["s"]), N


@pytest.mark.parametrize("call", ["run", "update"])
def test_large_table_recorded_before_anything_has_run(gpu, graphs, call):
    """A stream being captured allows no allocation: past 16,384 keys a first call is recorded
    all the same, without the cells that the two passes need."""
    N, W, H = 5000, 90, 70  # 25,200 keys
    cls, start = gpu.gen_maps_bernoulli(2, 1, N, W, H, 0.15)
    cfg = gpu.make_config(N, W, H, table_mode=gpu.TABLE_SHARED, map_mode=gpu.MAP_SHARED, lr=0.02, eps0=0.3,
                          episode_len=5, seed=3)
    stream = graphs.stream()

    def go(e):
        e.step_count = 0  # a replay draws what the recorded call drew
        if call == "run":
            e.run_fused(2)
        else:
            e.select(fetch=False)
            e.step()
            e.update()

    with gpu.Engine(cfg, 0) as want, gpu.Engine(cfg, 0) as eng:
        for e in (want, eng):
            e.set_maps(cls, start)
            assert e.lib.crl_set_stream(e.h, stream) == 0
        graph = graphs.record(stream, lambda: go(eng))
        for _ in range(3):
            graphs.replay(graph, stream)
            go(want)
            assert np.array_equal(want.q_get(0), eng.q_get(0))
            assert np.array_equal(want.get_state()["s"], eng.get_state()["s"])
            for e in (want, eng):  # eager work between the replays, which allocates the cells
                e.step_count = 7
                e.run_fused(3)
        assert np.array_equal(want.q_get(0), eng.q_get(0))
        for e in (want, eng):
            assert e.lib.crl_set_stream(e.h, None) == 0
        graphs.destroy(graph)
    graphs.destroy_stream(stream)


@pytest.mark.parametrize("N,steps", [(8192, 16), (8193, 14), (16385, 12), (32769, 10), (49153, 9)])
def test_calls_on_either_side_of_the_shortest_one_launch_call(gpu, oracle, N, steps):
    W, H = 24, 21
    cls, start = gpu.gen_maps_bernoulli(9, 1, N, W, H, 0.12, 0.03)
    cfg = gpu.make_config(N, W, H, table_mode=gpu.TABLE_SHARED, map_mode=gpu.MAP_SHARED, lr=0.003, eps0=0.3,
                          episode_len=30, seed=4)
    with gpu.Engine(cfg, 0) as eng:
        eng.set_maps(cls, start)
        assert eng.fused_kernel_info(steps)["name"].startswith("k_shared_persist")
        assert eng.fused_kernel_info(steps - 1)["name"] == "k_shared_act+k_reduce_owners"
        for n in (steps, steps - 1, steps):
            eng.run_fused(n)
        q, st = eng.q_get(0), eng.get_state()
    Q = np.zeros((1, W * H, 4), np.float32)
    ost = oracle.new_state(cfg, start)
    oracle.run(cfg, cls, None, start, Q, ost, 0, 3 * steps - 1)
    assert np.array_equal(q, Q[0]) and np.array_equal(st["s"], ost["s"])


@pytest.mark.parametrize("first,recorded", [(60, 6), (6, 60), (60, 60), (6, 6)])
def test_calls_of_any_length_are_recorded_once_one_has_run(gpu, graphs, first, recorded):
    """Short calls take two launches to a step, long ones one launch in all: what either needs is
    there after the first call of any length."""
    N, W, H = 3000, 16, 16
    cls, start = gpu.gen_maps_bernoulli(9, 1, N, W, H, 0.12, 0.03)
    cfg = gpu.make_config(N, W, H, table_mode=gpu.TABLE_SHARED, map_mode=gpu.MAP_SHARED, lr=0.003, eps0=0.3,
                          episode_len=30, seed=4)
    stream = graphs.stream()
    with gpu.Engine(cfg, 0) as want, gpu.Engine(cfg, 0) as eng:
        for e in (want, eng):
            e.set_maps(cls, start)
            assert e.lib.crl_set_stream(e.h, stream) == 0
            e.run_fused(first)
            e.step_count = 0
        names = [eng.fused_kernel_info(n)["name"] for n in (6, 60)]
        assert names == ["k_shared_act+k_reduce_owners", "k_shared_persist<4,1,folded>"]
        graph = graphs.record(stream, lambda: eng.run_fused(recorded))
        for _ in range(3):
            graphs.replay(graph, stream)
            want.step_count = 0
            want.run_fused(recorded)
            assert np.array_equal(want.q_get(0), eng.q_get(0))
            assert np.array_equal(want.get_state()["s"], eng.get_state()["s"])
            for e in (want, eng):
                e.step_count = 9
                e.run_fused(first)
        assert np.array_equal(want.q_get(0), eng.q_get(0))
        for e in (want, eng):
            assert e.lib.crl_set_stream(e.h, None) == 0
        graphs.destroy(graph)
    graphs.destroy_stream(stream)


@pytest.mark.parametrize("W,H", [(40, 30), (90, 70)])
@pytest.mark.parametrize("call", ["run", "update"])
def test_recorded_calls_keep_the_buffers_they_were_recorded_with(gpu, graphs, call, W, H):
    """A larger td_update between two replays needs larger buffers than the recorded launches have."""
    N = 5000
    cls, start = gpu.gen_maps_bernoulli(2, 1, N, W, H, 0.15)
    cfg = gpu.make_config(N, W, H, table_mode=gpu.TABLE_SHARED, map_mode=gpu.MAP_SHARED, lr=0.02, eps0=0.3,
                          episode_len=5, seed=3)
    stream = graphs.stream()
    rng = np.random.default_rng(W)
    small, large, larger = (transitions(rng, W * H, 4, n) for n in (6000, 40000, 90000))

    def go(e):
        e.step_count = 0
        if call == "run":
            e.run_fused(2)
        else:
            e.select(fetch=False)
            e.step()
            e.update()

    with gpu.Engine(cfg, 0) as want, gpu.Engine(cfg, 0) as eng:
        for e in (want, eng):
            e.set_maps(cls, start)
            assert e.lib.crl_set_stream(e.h, stream) == 0
            e.td_update(0, *small)
            go(e)
        graph = graphs.record(stream, lambda: go(eng))
        for batch in (small, large, larger):
            for e in (want, eng):
                e.td_update(0, *batch)
            graphs.replay(graph, stream)
            go(want)
            assert np.array_equal(want.q_get(0), eng.q_get(0))
            assert np.array_equal(want.get_state()["s"], eng.get_state()["s"])
        for e in (want, eng):
            assert e.lib.crl_set_stream(e.h, None) == 0
        graphs.destroy(graph)
    graphs.destroy_stream(stream)


@pytest.mark.parametrize("items", [
    lambda v: v,                                                   # exact ints, floats, bools and tuples
    lambda v: tuple(v),
    lambda v: [list(x) if isinstance(x, tuple) else x for x in v],
    lambda v: [tuple(np.int64(k) for k in x) if isinstance(x, tuple) else np.float64(x) if isinstance(x, float) else x
               for x in v],
])
def test_update_batch_takes_any_sequence_of_numbers(gpu, items):
    import os
    import sys
    sys.path.insert(0, os.path.join(os.path.dirname(gpu.__file__), "lib"))
    import cudarl_core
    s, s2 = [(1, 2), (0, 0), (1, 2)], [(2, 2), (0, 1), (2, 2)]
    args = (s, [0, 3, 0], [0.5, -1.0, 0.25], s2, [False, True, False])
    ref = cudarl_core.CudaQLearning(4, 3, 4)
    ref.update_batch(*args)
    q = cudarl_core.CudaQLearning(4, 3, 4)
    q.update_batch(*[items(v) for v in args])
    table = q.get_q_table()
    assert isinstance(table, list) and len(table) == 48 and table == ref.get_q_table()
    assert table[(2 * 4 + 1) * 4] == np.float32(np.float32(0.1) * np.float32(0.5)) + np.float32(np.float32(0.1) * np.float32(0.25))
    with pytest.raises(TypeError):
        q.update_batch(s, ["x", 3, 0], [0.5, -1.0, 0.25], s2, [False, True, False])
    with pytest.raises(TypeError):
        q.update_batch(s, [1 << 40, 3, 0], [0.5, -1.0, 0.25], s2, [False, True, False])
    with pytest.raises(RuntimeError, match="Inconsistent"):
        q.update_batch(s, [3, 0], [0.5, -1.0, 0.25], s2, [False, True, False])
    assert q.get_q_table() == table
