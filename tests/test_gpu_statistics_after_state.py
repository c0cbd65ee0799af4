"""Episode statistics that go out with the state for a caller who reads them after it: in every order of
calls that change the state, the statistics or the page they lie in, against an engine that is asked for its
statistics alone."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

STATS = ("last_return", "last_length", "return_sum", "length_sum")


def engines(gpu, N, **kw):
    W, H = 6, 5
    cls, start = gpu.gen_maps_bernoulli(5, N, N, W, H, 0.1, 0.05)
    cfg = gpu.make_config(N, W, H, episode_len=7, eps0=0.4, seed=9, track_returns=1, **kw)
    out = [gpu.Engine(cfg, 0), gpu.Engine(cfg, 0)]
    for e in out:
        e.set_maps(cls, start)
    return out


def check(want, eng):
    a, b = want.episode_stats(), eng.episode_stats()
    for k in STATS:
        assert np.array_equal(a[k], b[k]), k


@pytest.mark.parametrize("N", [1, 65, 4099, 130001])  # (the last: state and statistics together past what goes through pinned memory)
def test_in_every_order(gpu, N):
    want, eng = engines(gpu, N)
    with want, eng:
        for k in range(16):
            for e in (want, eng):
                e.run_fused(5)
            if k != 3:
                eng.get_state()
            if k == 5:
                eng.q_get(0, 1)  # (takes the page)
            if k == 6:
                eng.select()     # (so does this)
            if k == 7:
                for e in (want, eng):
                    e.reset(0, 1)
            if k in (8, 9):
                acts = np.zeros(N, np.int32)
                for e in (want, eng):
                    e.step(acts)
                    e.update()
            if k == 10:
                eng.get_state()
            if k != 4:           # (nobody asks: it stops, and starts again)
                check(want, eng)
            if k == 11:
                check(want, eng)
                assert np.array_equal(want.get_state()["s"], eng.get_state()["s"])
        assert np.array_equal(want.q_get(0, N), eng.q_get(0, N))


def test_after_the_replay_of_a_recorded_call(gpu, graphs):
    """A replay moves statistics without a call of the engine."""
    want, eng = engines(gpu, 300)
    stream = graphs.stream()

    def call(e):
        e.step_count = 0
        e.run_fused(9)

    with want, eng:
        for e in (want, eng):
            assert e.lib.crl_set_stream(e.h, stream) == 0
            call(e)
            e.get_state()
            e.episode_stats()
        graph = graphs.record(stream, lambda: call(eng))
        for _ in range(3):
            eng.get_state()
            graphs.replay(graph, stream)
            call(want)
            check(want, eng)
        for e in (want, eng):
            assert e.lib.crl_set_stream(e.h, None) == 0
        graphs.destroy(graph)
    graphs.destroy_stream(stream)
