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


def test_batches_beyond_one_gather_launch(nsg):
    """18 draws of the one sample in range: the step's loss is that sample's"""
    x, t = rand_inputs(51, 2)
    with nsg.Network(16, max_batch=18, seed=3) as net:
        for b in range(2):
            net.add_sample(x[b].reshape(-1, 9), t[b].reshape(-1, 6))
        want = net.eval(1, 1)
        got = net.train(1, batch=18, lr=1e-4, seed=5, first=1, count=1)[0]
    # 18 equal sums of 24576 terms in FP64
    assert abs(got - want) <= 1e-12 * want


def test_non_finite_loss_leaves_the_parameters_of_the_last_good_step(nsg):
    """the steps after a non-finite loss run, but change nothing: parameters, moments and step count
    are those of a run that stops there"""
    x, t = rand_inputs(52, 2)
    bad = t[1].copy()
    bad[3, 2, 1, 4] = np.inf

    def network():
        net = nsg.Network(16, seed=4)
        net.add_sample(x[0].reshape(-1, 9), t[0].reshape(-1, 6))
        net.add_sample(x[1].reshape(-1, 9), bad.reshape(-1, 6))
        return net

    steps, seed = 12, 0
    while True:  # a seed whose first draws are finite
        seed += 1
        with network() as net:
            with pytest.raises(nsg.NSGError) as e:
                net.train(steps, lr=1e-3, seed=seed)
            k = int(str(e.value).rsplit(" ", 1)[1])
            if 0 < k < steps - 2:
                net.train(2, lr=1e-3, seed=9, first=0, count=1)
                got = net.get_params()
                break
    with network() as net:
        assert np.isfinite(net.train(k, lr=1e-3, seed=seed)).all()
        net.train(2, lr=1e-3, seed=9, first=0, count=1)
        assert np.array_equal(net.get_params(), got)
