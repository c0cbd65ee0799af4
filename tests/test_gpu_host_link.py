"""What goes between host and kernels through pinned memory: actions in, actions, state and
tables out, at the sizes where the way they take changes (one env, one and several
workgroups, past the size that goes through pinned memory at all), and the state copy that
the step kernel keeps while the state is read after every step."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

NAMES = ("s", "ep_step", "episode", "reward", "done", "action")


def same(a, b):
    return all(np.array_equal(a[k], b[k]) for k in NAMES)


@pytest.mark.parametrize("N", [1, 2, 64, 65, 256, 257, 4099, 240001])
def test_rounds_with_the_state_read_in_every_order(gpu, N):
    W, H = 6, 5
    cls, start = gpu.gen_maps_bernoulli(5, N, N, W, H, 0.1, 0.05)
    cfg = gpu.make_config(N, W, H, episode_len=7, eps0=0.4, seed=9)
    with gpu.Engine(cfg, 0) as want, gpu.Engine(cfg, 0) as eng:
        want.set_maps(cls, start)
        eng.set_maps(cls, start)
        assert same(want.get_state(), eng.get_state())
        for k in range(12):
            want.run_fused(1)
            # actions through the host, or left on the device
            eng.step(eng.select() if k % 3 != 2 else (eng.select(fetch=False), None)[1])
            if k not in (4, 5, 8):  # read after every step but these: the copy stops and starts again
                if k == 6:
                    eng.q_get(0, 1)  # (takes the page that held the copy)
                assert same(want.get_state(), eng.get_state()), k
            eng.update()
            if k in (1, 7):  # the update leaves the state as it is
                assert same(want.get_state(), eng.get_state()), k
        assert np.array_equal(want.q_get(0, N), eng.q_get(0, N))
        eng.reset(0, 1)
        want.reset(0, 1)
        assert same(want.get_state(), eng.get_state())


def test_state_written_by_the_caller_is_what_the_next_read_returns(gpu):
    """Views of the state are out: no copy of it may be handed out in its place."""
    hip = C.CDLL("libamdhip64.so")
    N = 70
    mine = np.full(N, 7, np.int32)
    with gpu.Engine(gpu.make_config(N, 6, 5, seed=1), 0) as eng:
        eng.set_maps(np.zeros((N, 30), np.uint8), np.arange(N, dtype=np.int32) % 30)
        for _ in range(3):
            eng.step(np.zeros(N, np.int32))
            eng.get_state()
        view = eng.device_ptr(0)
        eng.step(np.zeros(N, np.int32))
        assert hip.hipMemcpy(C.c_void_p(view), C.c_void_p(mine.ctypes.data), C.c_size_t(4 * N), 1) == 0  # host to device
        assert np.array_equal(eng.get_state()["s"], mine)


@pytest.mark.parametrize("which,key", [(0, "s"), (1, "ep_step"), (2, "episode"), (3, "reward")])
def test_state_written_through_a_pointer_taken_after_the_step(gpu, which, key):
    """The step has left a copy of the state already when the pointer is asked for."""
    hip = C.CDLL("libamdhip64.so")
    N = 70
    mine = np.full(N, 7, np.float32 if key == "reward" else np.int32)
    with gpu.Engine(gpu.make_config(N, 6, 5, seed=1), 0) as eng:
        eng.set_maps(np.zeros((N, 30), np.uint8), np.arange(N, dtype=np.int32) % 30)
        for _ in range(3):
            eng.step(np.zeros(N, np.int32))
            eng.get_state()
        eng.step(np.zeros(N, np.int32))
        view = eng.device_ptr(which)
        for value in (7, 9):  # ... and once more through the pointer that is out
            mine[:] = value
            eng.sync()
            assert hip.hipMemcpy(C.c_void_p(view), C.c_void_p(mine.ctypes.data), C.c_size_t(4 * N), 1) == 0
            assert np.array_equal(eng.get_state()[key], mine)
        eng.step(np.zeros(N, np.int32))
        assert eng.get_state()["ep_step"][0] == (10 if key == "ep_step" else 5)


@pytest.mark.parametrize("recorded", ["run", "step", "reset"])
def test_state_after_the_replay_of_a_recorded_call(gpu, graphs, recorded):
    """A replay moves the state without a call of the engine: no copy that an earlier step
    left may be handed out."""
    N, W, H = 300, 9, 7
    cls, start = gpu.gen_maps_bernoulli(3, N, N, W, H, 0.1, 0.02)
    cfg = gpu.make_config(N, W, H, eps0=0.4, episode_len=11, seed=5)
    rng = np.random.default_rng(1)
    stream = graphs.stream()

    def call(e):
        e.step_count = 0  # a replay draws what the recorded call drew
        if recorded == "run":
            e.run_fused(3)
        elif recorded == "step":
            e.select(fetch=False)
            e.step()
        else:
            e.reset(0, N)

    with gpu.Engine(cfg, 0) as want, gpu.Engine(cfg, 0) as eng:
        for e in (want, eng):
            e.set_maps(cls, start)
            assert e.lib.crl_set_stream(e.h, stream) == 0
        graph = graphs.record(stream, lambda: call(eng))
        eng.reset(0, N)
        for _ in range(3):
            for _ in range(3):
                acts = rng.integers(0, 4, N).astype(np.int32)
                for e in (want, eng):
                    e.step(acts)
                assert same(want.get_state(), eng.get_state())
            acts = rng.integers(0, 4, N).astype(np.int32)
            for e in (want, eng):
                e.step(acts)
            graphs.replay(graph, stream)
            call(want)
            assert same(want.get_state(), eng.get_state())
        assert np.array_equal(want.q_get(0, N), eng.q_get(0, N))
        for e in (want, eng):
            assert e.lib.crl_set_stream(e.h, None) == 0
        graphs.destroy(graph)
    graphs.destroy_stream(stream)


def test_actions_may_be_overwritten_once_step_has_returned(gpu):
    N = 5000
    acts = np.zeros((20, N), np.int32)
    rng = np.random.default_rng(0)
    acts[:] = rng.integers(0, 4, acts.shape)
    cls = np.zeros((N, 99), np.uint8)
    start = np.full(N, 49, np.int32)
    with gpu.Engine(gpu.make_config(N, 11, 9, seed=1), 0) as eng:
        eng.set_maps(cls, start)
        buf = np.empty(N, np.int32)
        for a in acts:
            buf[:] = a
            eng.step(buf)
            buf[:] = -1
        st = eng.get_state()
    x, y = np.full(N, 5), np.full(N, 4)
    for a in acts:
        x = np.clip(x + (a == 1) - (a == 3), 0, 10)
        y = np.clip(y + (a == 2) - (a == 0), 0, 8)
    assert np.array_equal(st["s"], y * 11 + x)


def test_pages_grow_while_earlier_calls_still_read_them(gpu, oracle):
    """Batches of growing and shrinking size one after the other, without a wait between: four
    pages of a small size, two of a large one, all of one block."""
    W, H, A = 30, 20, 4
    S = W * H
    rng = np.random.default_rng(2)
    sizes = [1, 300, 900, 341, 342, 1025, 10922, 10923, 5, 40000, 3, 3, 3, 131072, 1500, 262144, 7, 262145, 64, 64, 64, 64, 64]
    want = rng.normal(0, 1, S * A).astype(np.float32)
    cfg = gpu.make_config(1, W, H, n_actions=A, table_mode=gpu.TABLE_SHARED, map_mode=gpu.MAP_SHARED, lr=1e-3)
    with gpu.Engine(cfg, 0) as eng:
        eng.q_set(0, want)
        batches = [(rng.integers(0, S, n), rng.integers(0, A, n), rng.normal(0, 1, n).astype(np.float32),
                    rng.integers(0, S, n), (rng.random(n) < 0.2).astype(np.uint8)) for n in sizes]
        for b in batches:
            eng.td_update(0, *b)
        for b in batches:
            oracle.td_update_batch(want, S, A, *b, 1e-3, 0.99, 0)
        assert np.array_equal(eng.q_get(0).reshape(-1), want)


def test_calls_that_take_host_data_are_refused_under_capture(gpu):
    """Their kernels read pages that are taken in turn: a replay would read another call's."""
    import torch
    cfg = gpu.make_config(8, 5, 5, table_mode=gpu.TABLE_SHARED, map_mode=gpu.MAP_SHARED)
    one = np.zeros(8, np.int32)
    stream = torch.cuda.Stream()
    with gpu.Engine(cfg, 0) as eng:
        assert eng.lib.crl_set_stream(eng.h, C.c_void_p(stream.cuda_stream)) == 0
        eng.td_update(0, one, one, np.ones(8, np.float32), one, one.astype(np.uint8))
        before = eng.q_get(0).copy()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.stream(stream):
            graph.capture_begin()
            for call in (lambda: eng.td_update(0, one, one, np.ones(8, np.float32), one, one.astype(np.uint8)),
                         lambda: eng.step(one)):
                with pytest.raises(gpu.CrlError, match="captured"):
                    call()
            graph.capture_end()
        assert np.array_equal(eng.q_get(0), before)
        eng.step(one)
        assert eng.lib.crl_set_stream(eng.h, None) == 0
