"""Refusals of the epilogue's gradient that need no device: they are raised before any kernel could run."""
import pytest
import torch

from approxtrain_amd import functors


@pytest.mark.parametrize("activation", ["sigmoid", "Relu", 1])
def test_unknown_activation_is_refused(activation):
    grad = torch.zeros(2, 3)
    with pytest.raises(ValueError, match="activation"):
        functors.epilogue_grad(grad, grad, True, activation)
