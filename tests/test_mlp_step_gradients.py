"""MLP.step gives its kernel tables of one entry per parameter: too few gradients are refused."""
import pytest
import torch


@pytest.mark.parametrize("weights,biases", [(3, 2), (3, 0), (0, 0)])
def test_missing_gradients_are_refused(weights, biases):
    from opengate_amd.learn.mlp import MLP

    net = MLP([8, 256, 256, 6], device="cpu")
    dW, db = [torch.zeros_like(w) for w in net.W], [torch.zeros_like(b) for b in net.b]
    with pytest.raises(RuntimeError, match="every weight and bias"):
        net.step(dW[:weights], db[:biases])
    assert net.t == 0
