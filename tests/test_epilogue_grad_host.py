"""Refusals of the epilogue's gradient that need no device: they are raised before any kernel could run."""
import pytest
import torch

from approxtrain_amd import functors, load_library


@pytest.mark.parametrize("activation", ["sigmoid", "Relu", 1])
def test_unknown_activation_is_refused(activation):
    grad = torch.zeros(2, 3)
    with pytest.raises(ValueError, match="activation"):
        functors.epilogue_grad(grad, grad, True, activation)


@pytest.mark.parametrize("shape", [(2, 2), (1, 3), (3,), (2, 3, 1), (3, 2), (4, 3)])
def test_output_of_another_shape_is_refused(shape):
    with pytest.raises(ValueError, match="shape"):
        functors.epilogue_grad(torch.zeros(2, 3), torch.zeros(shape), True, "relu")


@pytest.mark.parametrize("cols,shortest", [(1, 256), (16, 256), (17, 128), (32, 128), (33, 64), (4096, 64)])
def test_one_slab_needs_no_workspace(cols, shortest):
    """Rows that one workgroup adds go to the bias gradient at once: nothing to reduce, nothing to allocate."""
    query = load_library().amsim_epilogue_grad_workspace_bytes
    assert query(1, cols) == 0 and query(shortest, cols) == 0
    assert query(shortest + 1, cols) == 2 * cols * 4


@pytest.mark.parametrize("rows,cols", [(1, 1 << 30), (1 << 44, 3), (1 << 62, 4)])
def test_extents_beyond_the_grid_are_refused(rows, cols):
    lib = load_library()
    assert lib.amsim_epilogue_grad_workspace_bytes(rows, cols) == 0
    # (act NONE without a bias gradient: an accepted call has nothing to launch)
    assert lib.amsim_epilogue_grad_f32(None, None, rows, cols, 0, None, None, None, 0, None) == 6
    assert lib.amsim_epilogue_grad_f32(None, None, 1 << 20, 1 << 20, 0, None, None, None, 0, None) == 0


@pytest.mark.parametrize("rows,cols", [(0, 3), (3, 0), (0, 0)])
@pytest.mark.parametrize("act", [0, 1])
def test_empty_gradients_are_refused_at_the_boundary(rows, cols, act):
    """As the header says (functors.epilogue_grad answers them itself)."""
    assert load_library().amsim_epilogue_grad_f32(None, None, rows, cols, act, None, None, None, 0, None) == 1
