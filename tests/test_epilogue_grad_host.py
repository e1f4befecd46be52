"""Refusals of the epilogue's gradient that need no device: they are raised before any kernel could run."""
import pytest
import torch

from approxtrain_amd import functors


@pytest.mark.parametrize("activation", ["sigmoid", "Relu", 1])
def test_unknown_activation_is_refused(activation):
    grad = torch.zeros(2, 3)
    with pytest.raises(ValueError, match="activation"):
        functors.epilogue_grad(grad, grad, True, activation)


@pytest.mark.parametrize("shape", [(2, 2), (1, 3), (3,), (2, 3, 1), (3, 2), (4, 3)])
def test_output_of_another_shape_is_refused(shape):
    with pytest.raises(ValueError, match="shape"):
        functors.epilogue_grad(torch.zeros(2, 3), torch.zeros(shape), True, "relu")
