"""The predictor's kernels at the edges of their tiles: gradients of 1 to 300
rows (16-row tiles, 64-row sums, 128-step product loops over the rows, and
what is left over) against the fp64 restatement, and predictions on both sides
of 4096 nodes, from where a wave takes two, against the plain forward pass."""
import numpy as np
import pytest

import mlp_ref as M
import oracle as O
import spz

pytestmark = pytest.mark.gpu

# fp32 accumulation on the device, fp64 on the CPU, the same bf16 rounding
# points: a value next to a rounding point may fall to its other side
FWD_ATOL = 2e-3
GRAD_REL_L2 = 1e-2


@pytest.fixture(scope="module", params=[4, 5])
def solver(request):
    w = request.param
    with spz.Solver(width=w, frontier_target=16) as s:
        s.mlp_init(3)
        base = np.stack([O.walk(w, 3 + i % 70, 8_700_000 + i) for i in range(300)])
        yield s, base


@pytest.mark.parametrize("n", [1, 15, 16, 17, 63, 64, 65, 127, 128, 129, 143, 300])
def test_gradient(solver, n):
    s, base = solver
    print("gradient", n, flush=True)
    b = base[:n]
    h = s.eval_h(b)
    thr = (h + 2 * (np.arange(n) % 5)).astype(np.int32)
    tgt = np.linspace(0.0, 30.0, n).astype(np.float32)
    loss, g = s.mlp_grad(b, thr, tgt)
    lref, gref = M.grad(s.mlp_get_params(), M.features(b, thr, h), tgt)
    assert abs(loss - lref) <= 1e-3 * max(1.0, lref)
    assert np.linalg.norm(g - gref) <= GRAD_REL_L2 * np.linalg.norm(gref)


@pytest.mark.parametrize("n", [1, 2, 4095, 4096, 4097])
def test_prediction(solver, n):
    s, base = solver
    print("prediction", n, flush=True)
    b = base[np.arange(n) % len(base)]
    thr = (s.eval_h(b) + 2 * (np.arange(n) // len(base))).astype(np.int32)
    pred = s.mlp_predict(b, thr)
    for k in (0, 7, 15):
        y = s.mlp_forward(b, thr + 2 * k)
        assert np.max(np.abs(pred[:, k] - y)) <= FWD_ATOL * max(1.0, float(np.max(np.abs(y))))
