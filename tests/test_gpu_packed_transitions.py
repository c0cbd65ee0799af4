"""Transitions cross the link in 8 bytes where a key has 16 bits, in 12 above: both sides of that line, at
the last keys, with actions outside the table, states outside the map and calls of several pieces.
Bit for bit against the oracle: every sum has a stated order."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

INT = np.iinfo(np.int32)


def transitions(rng, S, A, n):
    s, s2 = rng.integers(0, S, n), rng.integers(0, S, n)
    edge = rng.random(n) < 0.2
    s[edge], s2[edge] = S - 1, S - 1
    a = rng.integers(0, A, n)
    a[edge] = A - 1
    outside = rng.random(n) < 0.05
    a[outside] = rng.choice([-1, A, 0xffff, 0x10000, INT.min, INT.max], int(outside.sum()))
    s[-1], a[-1] = S - 1, A - 1  # the last key of the table
    return s, a, rng.normal(0, 1, n).astype(np.float32), s2, (rng.random(n) < 0.3).astype(np.uint8) * 3


# keys: 4, 65,532 and 65,520, the most of one word; 65,536, the first of two
@pytest.mark.parametrize("W,H,A", [(1, 1, 4), (127, 129, 4), (91, 90, 8), (128, 128, 4), (64, 128, 8)])
@pytest.mark.parametrize("n", [1, 257, 1025, 65536, (1 << 18) + 1])
def test_both_forms(gpu, oracle, W, H, A, n):
    S, mode = W * H, n & 1
    rng = np.random.default_rng(n + S)
    cfg = gpu.make_config(1, W, H, n_actions=A, max_mode=mode, table_mode=gpu.TABLE_SHARED, map_mode=gpu.MAP_SHARED)
    want = rng.normal(0, 1, S * A).astype(np.float32)
    with gpu.Engine(cfg, 0) as eng:
        eng.q_set(0, want)
        for _ in range(3):
            b = transitions(rng, S, A, n)
            eng.td_update(0, *b)
            known = (b[1] >= 0) & (b[1] < A)
            oracle.td_update_batch(want, S, A, b[0], np.where(known, b[1], -1), *b[2:], 0.1, 0.99, mode)
        for which, state in ((0, S), (0, -1), (3, S), (3, 1 << 20), (3, INT.min)):  # refused, and nothing changed
            bad = [np.array(x) for x in b]
            bad[which][n // 2] = state
            with pytest.raises(gpu.CrlError):
                eng.td_update(0, *bad)
        if n <= 1024:
            keys, _ = eng.td_update_collect(0, *b)
            oracle.td_update_batch(want, S, A, b[0], np.where(known, b[1], -1), *b[2:], 0.1, 0.99, mode)
            assert S * A - 1 in keys
        assert np.array_equal(eng.q_get(0).reshape(-1), want)
