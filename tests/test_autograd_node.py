"""The native autograd node of a small loss (csrc/host/fs_autograd.cpp): what PyTorch asks of a node besides its
backward pass."""
import ctypes
from types import SimpleNamespace

import pytest
import torch
from torch._dynamo import compiled_autograd

from flash_sinkhorn_amd import _native, _small


class Ask(_small._Ask):
    """Stands for the gradient of a solve: 2 x, 3 y and multiples of what the node has saved behind them."""

    def __init__(self):
        super().__init__(None, None)

    def __call__(self, grad_out, tensors, need):
        x, y, pots = tensors[0], tensors[1], tensors[7]
        made = 2 * x * grad_out, 3 * y * grad_out, pots[:3] * grad_out, pots[3:] * grad_out
        return tuple(t if wanted else None for t, wanted in zip(made, need))


def node_loss(x, y, a, b, pots):
    form = _small.Problem()
    # (in double precision the node leaves its gradients to Python)
    saved = [x, y, x.detach(), y.detach(), None, None, torch.zeros(8, dtype=torch.uint8), pots]
    return _native.attach(torch.zeros(()), a, b, saved, ctypes.addressof(form), ctypes.sizeof(form), 0, Ask())


# Compiled autograd records a backward pass: the node was refused there ("compiled_args not implemented").  The second and third
# pass take the graph that the first one left.
@pytest.mark.parametrize("need", [(True, True, False, False), (False, True, None, None), (True, False, True, False),
                                  (True, False, None, True), (False, False, True, True)])
def test_compiled_autograd(need):
    gen = torch.Generator().manual_seed(1)
    for _ in range(3):
        given = [None if w is None else torch.randn(s, dtype=torch.float64, generator=gen).requires_grad_(w)
                 for s, w in zip(((3, 2), (4, 2), (3,), (3,)), need)]
        pots = torch.randn(6, dtype=torch.float64, generator=gen)
        leaves = [t for t in given if t is not None and t.requires_grad]

        def gradients():
            for t in leaves:
                t.grad = None
            x, y, a, b = (t if t is None else t * 1.5 for t in given)  # (not leaves)
            (2.0 * node_loss(x, y, a, b, pots)).backward()
            return [t.grad.clone() for t in leaves]

        want = gradients()
        with compiled_autograd._enable(lambda graph: graph):
            got = gradients()
        assert all(torch.equal(g, w) for g, w in zip(got, want))


# A loss of other tensors than those that a transform of functorch follows is refused as one of these is: a Function without rules
# for transforms is, and the native node says nothing of them.
def test_losses_inside_a_transform_are_refused(monkeypatch):
    x, y = torch.randn(3, 2, requires_grad=True), torch.randn(4, 2)
    monkeypatch.setattr(_small, "_solve_for", lambda *_, **__: pytest.fail("solved"))
    with pytest.raises(RuntimeError, match="functorch"):
        torch.func.grad(lambda s: s * _small.loss(SimpleNamespace(debias=False), x, y, None, None, False))(torch.tensor(2.0))


@pytest.mark.gpu
@pytest.mark.parametrize("weighted", [False, True])
def test_compiled_autograd_of_a_loss(weighted):
    from flash_sinkhorn_amd import SamplesLoss
    gen = torch.Generator(device="cuda").manual_seed(2)
    x, y = (torch.randn(2, n, 5, device="cuda", generator=gen).requires_grad_() for n in (70, 90))
    a, b = (torch.rand(2, n, device="cuda", generator=gen).add_(0.1).requires_grad_() for n in (70, 90))
    leaves = [x, y, a, b] if weighted else [x, y]

    def gradients():
        for t in leaves:
            t.grad = None
        out = SamplesLoss(debias=True)(*((a, x, b, y) if weighted else (x, y)))
        out.sum().backward()
        return [t.grad.clone() for t in leaves]

    want = gradients()
    with compiled_autograd._enable(lambda graph: graph):
        for _ in range(2):
            assert all(torch.equal(g, w) for g, w in zip(gradients(), want))
