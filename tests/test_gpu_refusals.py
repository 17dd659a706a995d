"""A bad board leaves the caller's outputs as they were: the C entry points
with outputs filled beforehand, where the host checks the boards and where the
device does, and the predictor's parameters after a refused training."""
import ctypes

import numpy as np
import pytest

import oracle as O
import spz

pytestmark = pytest.mark.gpu


def ptr(a, t):
    return a.ctypes.data_as(ctypes.POINTER(t))


@pytest.mark.parametrize("width", [4, 5])
@pytest.mark.parametrize("n,at", [(1, 0), (256, 255), (257, 0), (300, 256), (20000, 19999), (70000, 65536)])
def test_outputs_are_untouched(width, n, at):
    base = np.stack([O.walk(width, 5 + i % 60, 9_600_000 + i) for i in range(61)]).astype(np.uint8)
    b = base[np.arange(n) % 61].copy()
    b[at, [1, 2]] = b[at, [2, 1]]
    L, u8, i32, f32 = spz.lib(), ctypes.c_uint8, ctypes.c_int32, ctypes.c_float
    thr, tgt = np.full(n, 60, np.int32), np.linspace(0, 20, n).astype(np.float32)
    print("refusals", width, n, at, flush=True)
    with spz.Solver(width=width, frontier_target=16) as s:
        s.mlp_init(1)
        before = s.mlp_get_params()
        h, y, p = np.full(n, -77, np.int32), np.full(n, -7.5, np.float32), np.full((n, 16), -7.5, np.float32)
        g, loss = np.full(s.mlp_param_count(), -7.5, np.float32), np.full(1, -7.5, np.float32)
        ep = np.full(1, -7.5, np.float32)
        calls = [L.spz_eval_h(s._ctx, ptr(b, u8), n, ptr(h, i32))]
        if n <= spz.NOALLOC_MAX_BOARDS:
            calls.append(L.spz_eval_h_noalloc(s._ctx, ptr(b, u8), n, ptr(h, i32)))
        calls.append(L.spz_mlp_forward(s._ctx, ptr(b, u8), ptr(thr, i32), n, ptr(y, f32)))
        calls.append(L.spz_mlp_predict(s._ctx, ptr(b, u8), ptr(thr, i32), n, ptr(p, f32)))
        if n <= 20000:
            calls.append(L.spz_mlp_grad(s._ctx, ptr(b, u8), ptr(thr, i32), ptr(tgt, f32), n, ptr(loss, f32), ptr(g, f32)))
        calls.append(L.spz_mlp_train(s._ctx, ptr(b, u8), ptr(thr, i32), ptr(tgt, f32), n, 1, 64, 1e-3, 3, ptr(ep, f32)))
        assert calls == [-1] * len(calls)
        assert f"board {at} " in L.spz_last_error(s._ctx).decode()
        assert (h == -77).all()
        for out in (y, p, g, loss, ep):
            assert (out == -7.5).all()
        assert (s.mlp_get_params() == before).all()
        if n <= 300:
            res, ic = (spz._Result * n)(), np.full((n, 8), 77, np.uint64)
            ctypes.memset(res, 0x5a, ctypes.sizeof(res))
            assert L.spz_solve_batch(s._ctx, ptr(b, u8), n, 8, res, ptr(ic, ctypes.c_uint64)) == -1
            assert bytes(res) == b"\x5a" * ctypes.sizeof(res) and (ic == 77).all()
        # and the same call with the board put right
        b[at, [1, 2]] = b[at, [2, 1]]
        assert (s.eval_h(b) == np.array([O.manhattan(x) for x in base])[np.arange(n) % 61]).all()
