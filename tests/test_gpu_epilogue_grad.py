"""Gradient of the fused bias + ReLU epilogue: edges of the column tiles, of the rows per slab and of the slab count."""
import pytest
import torch

from approxtrain_amd import functors, layers

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,cols", [(1, 1), (3, 16), (255, 17), (256, 6), (257, 16), (129, 33), (64, 64), (65, 65),
                                       (1000, 513), (25600, 16), (140000, 70), (600001, 3)])
@pytest.mark.parametrize("act", ["relu", None])
@pytest.mark.parametrize("has_bias", [True, False])
def test_epilogue_grad(rows, cols, act, has_bias):
    gen = torch.Generator().manual_seed(rows * 1000 + cols)
    grad, out = torch.randn(rows, cols, generator=gen), torch.randn(rows, cols, generator=gen).relu_()
    z, b = functors.epilogue_grad(grad.cuda(), out.cuda(), has_bias, act)
    want = grad * (out > 0) if act == "relu" else grad
    assert torch.equal(z.cpu(), want)
    assert (b is None) == (not has_bias)
    if has_bias:
        # every 32-bit sum of n terms lies within n * 2^-24 * sum|terms|; slabs, chains and ways cut the n of
        # any one chain below 1024 (rows of a slab per chain + ways + slabs per chain)
        bound = 1024 * 2.0 ** -24 * want.double().abs().sum(0)
        assert ((b.cpu().double() - want.double().sum(0)).abs() <= bound).all()
        again = functors.epilogue_grad(grad.cuda(), out.cuda(), True, act)[1]
        assert torch.equal(b, again)


def test_infinite_gradient_of_a_masked_element_is_nan():
    grad = torch.tensor([[float("inf"), 1.0], [2.0, float("nan")]]).cuda()
    out = torch.tensor([[0.0, 1.0], [1.0, float("nan")]]).cuda()
    z, b = functors.epilogue_grad(grad, out, True, "relu")
    assert torch.equal(torch.isnan(z).cpu(), torch.tensor([[True, False], [False, True]]))
    assert torch.isnan(b).all()


@pytest.mark.parametrize("shape", [(0, 3), (2, 0, 70), (3, 0), (0,)])
@pytest.mark.parametrize("act", ["relu", None])
def test_empty_gradient(shape, act):
    grad = torch.empty(shape).cuda()
    z, b = functors.epilogue_grad(grad, torch.empty(shape).cuda(), True, act)
    assert z.shape == grad.shape and torch.equal(b.cpu(), torch.zeros(shape[-1]))


@pytest.mark.parametrize("rows,cols,act,calls", [(1, 1, None, 0), (80, 128, None, 0), (2047, 256, None, 0), (1023, 2048, None, 0),
                                                 (2048, 256, None, 1), (1024, 512, None, 1), (80, 128, "relu", 1), (2048, 256, "relu", 1)])
def test_small_gradients_of_a_bias_alone_stay_with_torch(monkeypatch, rows, cols, act, calls):
    seen = []
    library = functors.epilogue_grad_checked
    monkeypatch.setattr(functors, "epilogue_grad_checked", lambda *a: seen.append(a) or library(*a))
    gen = torch.Generator(device="cuda").manual_seed(rows + cols)
    grad, out = (torch.randn((rows, cols), device="cuda", generator=gen) for _ in range(2))
    with torch.no_grad():
        z, b = layers._epilogue_backward(grad, out, True, act)
    want = grad * (out > 0) if act == "relu" else grad
    assert torch.equal(z, want) and len(seen) == calls
    # (any order of the sum: n * 2^-24 * sum|terms|)
    assert ((b.double() - want.double().sum(0)).abs() <= rows * 2.0 ** -24 * want.double().abs().sum(0)).all()


def test_captured_bias_gradient_replays():
    """A captured pass stays with the library at every size: torch's sum over many blocks clears its
    counters by a recorded memset."""
    gen = torch.Generator(device="cuda").manual_seed(11)
    grad = torch.randn((2000, 256), device="cuda", generator=gen)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.no_grad(), torch.cuda.graph(graph):
        captured = layers._epilogue_backward(grad, None, True, None)[1]
    for i in range(4):
        grad.copy_(torch.randn((2000, 256), device="cuda", generator=gen))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(captured, functors.epilogue_grad(grad, None, True, None)[1]), i
        (grad * 2).sum(0)  # (eager work between the replays)
        torch.cuda.synchronize()


@pytest.mark.parametrize("rows,cols", [(25600, 16), (200704, 6), (401408, 16), (262144, 100), (50000, 600)])
def test_error_against_64_bits(rows, cols):
    """Positive terms, 100 slabs of rows and more: a slab's rounding errors average out over the slabs, so what is
    left is the one rounding of the result, at most 2^-24 of each column's sum."""
    gen = torch.Generator(device="cuda").manual_seed(rows)
    grad = torch.rand((rows, cols), device="cuda", generator=gen)
    want = grad.double().sum(0)
    got = functors.epilogue_grad(grad, None, True, None)[1].double()
    assert (got - want).norm() <= 2.0 ** -24 * want.norm()
