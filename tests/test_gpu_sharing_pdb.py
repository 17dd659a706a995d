"""Work sharing in the pattern-database search, whose parts of it are its own
(the taker computes its lookups from the board, the giver's cached sibling
values are voided): lengths and per-iteration counts equal the oracle's at the
edges of its range, and paths kept through lane exchange and mailboxes lead to
the goal.  And a single instance, whose iterations one workgroup restarts:
alone as in a batch, under every dispatch order, with heavy nodes split again."""
import numpy as np
import pytest

import oracle as O
import spz

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)


@pytest.fixture(scope="module")
def sets():
    with spz.Solver(width=5, heuristic=spz.H_PDB666, frontier_target=16) as s:
        s.build_pdb()
        O.pdb_set_tables(s.get_pdb(0), s.get_pdb(1))
    boards = [O.walk(5, d, 9_200_000 + d) for d in (0, 1, 40, 80, 96, 104, 110, 116)]
    say("oracle")
    return boards, [O.ida(b, heuristic="pdb") for b in boards]


def solver(**kw):
    s = spz.Solver(width=5, heuristic=spz.H_PDB666, **kw)
    s.build_pdb()
    return s


def check(res, expect):
    for k, (r, (opt, thr, cnt)) in enumerate(zip(res, expect)):
        assert (r.opt_len, r.thresholds, r.counts) == (opt, thr, cnt), k


def replay(board, moves):
    b = [int(x) for x in board]
    z = b.index(0)
    for d in moves:
        r, c = divmod(z, 5)
        r, c = r + (-1, 0, 0, 1)[d], c + (0, 1, -1, 0)[d]
        assert 0 <= r < 5 and 0 <= c < 5
        b[z], b[r * 5 + c] = b[r * 5 + c], 0
        z = r * 5 + c
    return b == list(range(25))


@pytest.mark.parametrize("kw", [dict(lanes=64, workgroup_size=64), dict(lanes=256), dict(lanes=1088, workgroup_size=64),
                                dict(lanes=1 << 20), dict(round_budget=1, lanes=4096),
                                dict(round_budget=9, frontier_target=1), dict(round_time_us=-1, lanes=2048),
                                dict(lds_stack_depth=8), dict(lookahead=False)],
                         ids=lambda k: "-".join(f"{a}={b}" for a, b in k.items()))
def test_sharing_matches_oracle(sets, kw):
    boards, expect = sets
    say("sharing, PDB", kw)
    with solver(record_paths=True, **kw) as s:
        res = s.solve(boards)
        check(res, expect)
        for b, r, moves in zip(boards, res, s.get_paths()):
            assert len(moves) == r.opt_len and replay(b, moves)


@pytest.mark.parametrize("kw", [dict(), dict(round_budget=3, lanes=2048), dict(lb_policy=spz.LB_PREVLOAD, resplit=2),
                                dict(lb_policy=spz.LB_LEARNED, resplit=1), dict(use_graph=False, frontier_target=7)],
                         ids=lambda k: "-".join(f"{a}={b}" for a, b in k.items()) or "default")
@pytest.mark.parametrize("paths", [False, True])
def test_alone_as_in_a_batch(sets, kw, paths):
    boards, expect = sets
    say("one instance, PDB", kw, paths)
    with solver(record_paths=paths, **kw) as s:
        if kw.get("lb_policy") == spz.LB_LEARNED:
            s.mlp_init(11)  # any parameters: the policy changes the schedule only
        for k, b in enumerate(boards):
            res = s.solve([b])
            check(res, expect[k:k + 1])
            if paths:
                moves = s.get_paths()[0]
                assert len(moves) == res[0].opt_len and replay(b, moves)
        check(s.solve(boards), expect)


@pytest.mark.parametrize("width", [4, 5])
def test_learned_order_alone_as_in_a_batch(width):
    """The learned order without tables, and its recorded paths."""
    boards = [O.walk(width, d, 9_300_000 + d) for d in (0, 1, 30, 46, 58)]
    expect = [O.ida(b) for b in boards]
    with spz.Solver(width=width, lb_policy=spz.LB_LEARNED, resplit=1, frontier_target=256, record_paths=True) as s:
        s.mlp_init(5)
        for k, b in enumerate(boards):
            check(s.solve([b]), expect[k:k + 1])
            assert len(s.get_paths()[0]) == expect[k][0]
        check(s.solve(boards), expect)
        assert [len(m) for m in s.get_paths()] == [e[0] for e in expect]


def test_logged_loads_are_the_counts():
    """With the root as the only frontier node, a sample's load is the count of
    its iteration.  4096 searches of one item each: waves run out of work and
    are fed all the time, and no node is lost or counted twice for its item."""
    n = 4096
    boards = np.stack([spz.gen_walk(4, 20 + i % 41, 9_400_000 + i) for i in range(n)])
    with spz.Solver(width=4, frontier_target=1, log_samples=200_000) as s:
        say("logged solve")
        res = s.solve(boards)
        b, thr, load = s.get_samples()
    # an iteration is logged when the next one starts
    want = {}
    for board, r in zip(boards, res):
        for t, c in list(zip(r.thresholds, r.counts))[:-1]:
            want.setdefault((board.tobytes(), t), []).append(c)
    assert len(load) == sum(len(v) for v in want.values())
    got = {}
    for x, t, l in zip(b, thr, load):
        got.setdefault((np.asarray(x, dtype=np.uint8).tobytes(), int(t)), []).append(int(l))
    assert got.keys() == want.keys()
    for k in want:
        assert sorted(got[k]) == sorted(want[k])


def test_a_large_logged_batch_runs_to_its_end():
    n = 4096
    boards = np.stack([spz.gen_walk(4, 20 + i * 60 // n, 9_500_000 + i) if i % 2 else spz.gen_random(4, 9_550_000 + i)
                       for i in range(n)])
    with spz.Solver(width=4, frontier_target=16) as s:
        say("plain solve")
        plain = [(r.opt_len, r.counts) for r in s.solve(boards)]
    with spz.Solver(width=4, frontier_target=16, log_samples=1_000_000) as s:
        say("logged solve")
        assert [(r.opt_len, r.counts) for r in s.solve(boards)] == plain
