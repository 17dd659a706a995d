"""The hipGraph of the search rounds is made once a solve has run six polls of
rounds: a solve of many short rounds replays it, a short one, one with the
graph off and one that times its kernels do not, and the statistics say which.
Lengths and counts are the oracle's on every path, several solves in a row."""
import pytest

import oracle as O
import spz

pytestmark = pytest.mark.gpu

MANY = dict(lanes=1024, round_budget=2)  # many rounds of two steps


@pytest.fixture(scope="module")
def sets():
    out = {}
    for w in (4, 5):
        boards = [O.walk(w, d, 9_100_000 + d) for d in (30, 40, 44)]
        out[w] = (boards, [O.ida(b) for b in boards])
    return out


@pytest.mark.parametrize("width", [4, 5])
@pytest.mark.parametrize("n", [1, 3])
@pytest.mark.parametrize("kw,replayed", [(MANY, True), (dict(MANY, use_graph=False), False),
                                         (dict(MANY, time_kernels=True), False), (dict(), False)],
                         ids=["graph", "off", "timed", "short"])
def test_replays(sets, width, n, kw, replayed):
    boards, expect = (x[-n:] for x in sets[width])
    print("graph replay", width, n, kw, flush=True)
    with spz.Solver(width=width, **kw) as s:
        for rep in range(3):
            for r, (opt, thr, cnt) in zip(s.solve(boards), expect):
                assert (r.opt_len, r.thresholds, r.counts) == (opt, thr, cnt)
            st = s.stats()
            assert (st["graph_replays"] > 0) == replayed, st
            assert st["graph"] == (0 if kw.get("time_kernels") or kw.get("use_graph") is False else 1)
