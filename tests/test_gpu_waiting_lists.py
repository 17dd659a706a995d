"""Waves without work wait on lists and are taken off them by waves that give
work.  With many small instances waves run out and are fed all the time, and
the log of samples slows the givers: a wave's list entry may be written over
soon after the wave is taken off.  The batch runs to its end, with the counts
of the search without the log, and the log's loads add up as ever."""
import numpy as np
import pytest

import spz

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [256, 2048])
def test_logged_batch_runs_to_its_end(n):
    boards = np.stack([spz.gen_walk(4, 20 + i * 60 // n, 8_900_000 + i) if i % 2 else spz.gen_random(4, 8_950_000 + i)
                       for i in range(n)])
    print("waiting lists", n, flush=True)
    with spz.Solver(width=4, frontier_target=16, lookahead=False) as s:
        plain = [(r.opt_len, r.counts) for r in s.solve(boards)]
    with spz.Solver(width=4, frontier_target=16, log_samples=2_000_000) as s:
        assert [(r.opt_len, r.counts) for r in s.solve(boards)] == plain
