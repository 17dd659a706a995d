"""A single instance has its iterations restarted, its lookahead asked for and
its queue published by one workgroup, a batch by three launches: each board
solved alone gives the oracle's result, as in a batch, under every dispatch
order, with heavy nodes split again, with paths and with rounds of a few
steps."""
import pytest

import oracle as O
import spz

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def sets():
    out = {}
    for w in (4, 5):
        boards = [O.walk(w, d, 8_800_000 + d) for d in (0, 1, 30, 46, 60)]
        out[w] = (boards, [O.ida(b) for b in boards])
    return out


@pytest.mark.parametrize("width", [4, 5])
@pytest.mark.parametrize("kw", [dict(), dict(lookahead=False), dict(round_budget=3, lanes=2048),
                                dict(lb_policy=spz.LB_PREVLOAD, resplit=2), dict(record_paths=True),
                                dict(use_graph=False, frontier_target=7)],
                         ids=lambda k: "-".join(f"{a}={b}" for a, b in k.items()) or "default")
def test_alone_as_in_a_batch(sets, width, kw):
    boards, expect = sets[width]
    print("one instance", width, kw, flush=True)
    with spz.Solver(width=width, **kw) as s:
        alone = [s.solve([b])[0] for b in boards]
        for res in (alone, s.solve(boards)):
            for r, (opt, thr, cnt) in zip(res, expect):
                assert (r.opt_len, r.thresholds, r.counts) == (opt, thr, cnt)
