"""Work sharing inside a search round (lanes of a wave take each other's open
nodes, waves without work are fed through mailboxes): it decides where nodes
are searched, never which, so lengths and per-iteration counts equal the
oracle's at the edges of its range -- one wave, one workgroup, a few waves on
many lists, more lanes than the device runs at once, rounds of a few steps,
and two contexts searching at the same time."""
import sys
import threading

import pytest

import oracle as O
import spz

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


@pytest.fixture(scope="module")
def sets():
    b4 = [O.walk(4, 30 + i % 25, 8_100_000 + i) for i in range(12)]
    b5 = [O.walk(5, 36 + i % 20, 8_200_000 + i) for i in range(6)]
    return {4: (b4, [O.ida(b) for b in b4]), 5: (b5, [O.ida(b) for b in b5])}


def check(res, expect):
    for r, (opt, thr, cnt) in zip(res, expect):
        assert (r.opt_len, r.thresholds, r.counts) == (opt, thr, cnt)


@pytest.mark.parametrize("width", [4, 5])
@pytest.mark.parametrize("kw", [dict(lanes=64, workgroup_size=64), dict(lanes=256), dict(lanes=1088, workgroup_size=64),
                                dict(lanes=1 << 20), dict(round_budget=1, lanes=4096), dict(round_budget=9, frontier_target=1),
                                dict(round_time_us=-1, lanes=2048), dict(lds_stack_depth=8)])
def test_sharing_matches_oracle(sets, width, kw):
    boards, expect = sets[width]
    say("sharing", width, kw)
    with spz.Solver(width=width, **kw) as s:
        check(s.solve(boards), expect)


@pytest.mark.parametrize("width", [4, 5])
def test_first_solution_drops_only_the_rest(sets, width):
    """First-solution mode drops the rest of every item of an instance once a
    goal is known: lengths and all counts but the last stay."""
    boards, expect = sets[width]
    with spz.Solver(width=width, mode=spz.MODE_FIRST, frontier_target=16) as s:
        for r, (opt, thr, cnt) in zip(s.solve(boards), expect):
            assert (r.opt_len, r.thresholds, r.counts[:-1]) == (opt, thr, cnt[:-1])
            assert r.counts[-1] <= cnt[-1]


def test_two_contexts_at_once(sets):
    """Rounds whose waves wait for work do not depend on a device of their
    own: two contexts, a thread each, search at the same time."""
    out = {}

    def work(width):
        with spz.Solver(width=width) as s:
            for _ in range(3):
                out[width] = s.solve(sets[width][0])

    ts = [threading.Thread(target=work, args=(w,)) for w in (4, 5)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    for w in (4, 5):
        check(out[w], sets[w][1])
