"""The training kernels of the wall-stress network at the edges of their batches:
one pair of groups, a half turn of a wave, exactly one fill of the product's
operands, one product more, and samples short of the batch; and the weights the
optimiser leaves for the next batch."""
import numpy as np
import pytest

from channel_rl_amd import WallNetwork
from oracle import mlp as om
from test_gpu_mlp import BLOCKS, _net_and_data

pytestmark = pytest.mark.gpu


# 2e-2 of a parameter block's norm: BF16 roundings that fall on the other side
# of a tie against the FP64 oracle, as for one batch in test_gpu_mlp.py; with few
# samples one such rounding weighs more, so at least 32 of them
@pytest.mark.parametrize("n", [32, 65, 96, 1024, 1056, 2077])
def test_gradients_at_batch_edges(gpu, n):
    net, p, norm, X, T = _net_and_data(4, n)
    g, loss = net.gradients(X, T)
    gr, lr = om.gradients(p, norm, X, T)
    assert abs(loss - lr) <= 1e-3 * lr
    for name, a, b in BLOCKS:
        e = np.linalg.norm(g[a:b] - gr[a:b]) / np.linalg.norm(gr[a:b])
        assert e <= 2e-2, (name, e)


# one sample has one order: three epochs of one call (the optimiser writes the
# next batch's operands) and three calls (operands rebuilt from the parameters)
# take the same steps, bit for bit, and so does the network they leave
def test_operands_follow_the_parameters(gpu):
    out = []
    for calls in (1, 3):
        net, _, _, X, T = _net_and_data(6, 1)
        for _ in range(calls):
            net.train(X, T, epochs=3 // calls, batch=32, lr=1e-2, seed=1)
        out.append((net.params()[0], net.forward(X)))
    assert np.isfinite(out[0][0]).all()
    for a, b in zip(*out):
        assert np.array_equal(a, b)
    assert not np.array_equal(out[0][0], WallNetwork(seed=6).params()[0])
