"""Backward kernels of the closure network over the shapes of their tile walk, against the closure
oracle (bar 2e-2 per layer, one bfloat16 rounding moved by FP32 order: tests/test_gpu_closure.py)."""
import numpy as np
import pytest

from conftest import rel
from test_gpu_closure import C, oracle_params, rand_inputs

pytestmark = pytest.mark.gpu


# weight-gradient blocks: 8 tiles for 256 blocks (idle blocks); 192; 432 (some blocks take two)
@pytest.mark.parametrize("N,B", [(16, 1), (32, 3), (48, 2)])
def test_gradients_over_the_tile_walk(nsg, N, B):
    x, t = rand_inputs(40 + N, B, N)
    with nsg.Network(N, max_batch=B, seed=6) as net:
        loss, g = net.loss_grad(x, t)
        again = net.loss_grad(x, t)
        params = oracle_params(net)
    assert again[0] == loss and np.array_equal(again[1], g)
    lo, go = C.loss_and_grads(params, x.astype(np.float64), t.astype(np.float64), emulate_bf16=True)
    assert abs(loss - lo) < 1e-3 * lo
    off = 0
    for l, (dW, db) in enumerate(go):
        for want in (dW, db):
            got = g[off:off + want.size].reshape(want.shape)
            off += want.size
            assert rel(got, want) < 2e-2, (l, want.shape)
