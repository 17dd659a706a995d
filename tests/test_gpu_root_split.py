"""The start of a solve: one workgroup splits an instance's root up to a
frontier of 16,384 nodes, the whole device beyond.  Lengths and per-iteration
counts are the oracle's on both sides of that line and at the split's edges --
a frontier of the root alone, no split level allowed, roots solved within the
split, more instances than the device holds workgroups of at once."""
import pytest

import oracle as O
import spz

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def sets():
    out = {}
    for w, seed in ((4, 8_300_000), (5, 8_400_000)):
        boards = [list(range(w * w))] + [O.walk(w, d, seed + d) for d in (1, 2, 9, 24, 40)]
        out[w] = (boards, [O.ida(b) for b in boards])
    return out


@pytest.mark.parametrize("width,heur", [(4, spz.H_MANHATTAN), (5, spz.H_MANHATTAN)])
@pytest.mark.parametrize("kw", [dict(frontier_target=1), dict(frontier_target=5), dict(max_split_depth=0),
                                dict(max_split_depth=1), dict(frontier_target=16384), dict(frontier_target=16385),
                                dict(frontier_target=16384, record_paths=True),
                                dict(frontier_target=16385, record_paths=True), dict(use_graph=False)],
                         ids=lambda k: "-".join(f"{a}={b}" for a, b in k.items()))
def test_split_matches_oracle(sets, width, heur, kw):
    boards, expect = sets[width]
    print("root split", width, kw, flush=True)
    with spz.Solver(width=width, heuristic=heur, **kw) as s:
        for n in (len(boards), 1, len(boards)):
            for r, (opt, thr, cnt) in zip(s.solve(boards[:n]), expect):
                assert (r.opt_len, r.thresholds, r.counts) == (opt, thr, cnt)


def test_many_instances(sets):
    boards, expect = sets[4]
    k = 200
    with spz.Solver(width=4, frontier_target=64) as s:
        for r, (opt, thr, cnt) in zip(s.solve(boards * k), expect * k):
            assert (r.opt_len, r.thresholds, r.counts) == (opt, thr, cnt)
