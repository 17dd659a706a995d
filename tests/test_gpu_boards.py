"""Boards are checked, packed and evaluated on the device, in pieces of 65,536
that pass through staging of 16 MB: values at the edges of a workgroup (256
boards), a piece and the staging, and a bad board refused with its index --
the lowest one -- and the outputs untouched, wherever it stands."""
import numpy as np
import pytest

import oracle as O
import spz

pytestmark = pytest.mark.gpu


def some(width, n):
    base = np.stack([O.walk(width, 5 + i % 60, 8_500_000 + i) if i % 2 else O.random_solvable(width, 8_600_000 + i)
                     for i in range(97)]).astype(np.uint8)
    return base[np.arange(n) % 97], np.array([O.manhattan(b) for b in base])[np.arange(n) % 97]


@pytest.mark.parametrize("width", [4, 5])
@pytest.mark.parametrize("n", [1, 2, 255, 256, 257, 65535, 65536, 65537, 900_001])
def test_values(width, n):
    b, h = some(width, n)
    print("boards", width, n, flush=True)
    with spz.Solver(width=width, frontier_target=16) as s:
        assert (s.eval_h(b) == h).all()
        if n <= spz.NOALLOC_MAX_BOARDS:
            assert (s.eval_h_noalloc(b) == h).all()


def test_values_beyond_staging():
    # 4,300,001 values do not fit the 16 MB of pinned results
    b, h = some(4, 4_300_001)
    with spz.Solver(width=4, frontier_target=16) as s:
        assert (s.eval_h(b) == h).all()


def bad_ones(width):
    n2 = width * width
    goal = np.arange(n2, dtype=np.uint8)
    swap, twice, high = goal.copy(), goal.copy(), goal.copy()
    swap[[1, 2]] = swap[[2, 1]]
    twice[3] = 4
    high[n2 - 1] = 255
    n2_itself = goal.copy()
    n2_itself[5] = n2
    return [swap, twice, high, n2_itself]


@pytest.mark.parametrize("width", [4, 5])
@pytest.mark.parametrize("n,at", [(1, (0,)), (256, (255,)), (300, (255, 256)), (20000, (19999,)), (70000, (65536, 69999)), (140000, (139999,))])
def test_bad_boards(width, n, at):
    b, h = some(width, n)
    rng = np.random.default_rng(1)
    with spz.Solver(width=width, frontier_target=16) as s:
        s.mlp_init(1)
        for bad in bad_ones(width):
            x = b.copy()
            for i in at:
                x[i] = bad
            calls = [lambda: s.eval_h(x)]
            if n <= spz.NOALLOC_MAX_BOARDS:
                calls += [lambda: s.eval_h_noalloc(x)]
            if n <= 300:
                thr = np.full(n, 40, dtype=np.int32)
                tgt = rng.random(n).astype(np.float32)
                calls += [lambda: s.mlp_forward(x, thr), lambda: s.mlp_predict(x, thr),
                          lambda: s.mlp_grad(x, thr, tgt), lambda: s.mlp_train(x, thr, tgt, epochs=1, batch=64),
                          lambda: s.solve(x)]
            for call in calls:
                with pytest.raises(spz.SpzError, match=f"board {at[0]} is not a solvable permutation"):
                    call()
        assert (s.eval_h(b) == h).all()
