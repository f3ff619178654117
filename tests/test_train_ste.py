"""ste's single pass against the plain expression y + (x - x.detach()): values, gradients of both orders, tangents,
batched transforms, tracing (CPU)."""
import numpy as np
import pytest
import torch
import torch.autograd.forward_ad as fwd

import lfm3_kv800_amd  # noqa: F401
from lfm3_kv800_amd.train import ste


def plain(x, fq):
    with torch.no_grad():
        y = fq(x)
    return y + (x - x.detach())


FQS = {"round": torch.round, "square": lambda t: t * t, "same": lambda t: t, "wide": lambda t: t.double() * 2,
       "broadcast": lambda t: torch.ones(2, *t.shape), "number": lambda t: 2.0}


def values(f, fq):
    return lambda x: (f(x, fq).to(torch.float32) ** 3).sum()


@pytest.mark.parametrize("fq", FQS.values(), ids=FQS.keys())
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_ste_derivatives(fq, dtype):
    out = []
    for f in (plain, ste):
        x = (torch.arange(-3.0, 3.0) * 0.7 + 0.1).to(dtype).requires_grad_()
        y = f(x, fq)
        g, = torch.autograd.grad((y ** 3).sum(), x, create_graph=True)
        gg, = torch.autograd.grad(g.sum(), x)
        with fwd.dual_level():
            d = fwd.unpack_dual(f(fwd.make_dual(x.detach(), torch.ones_like(x)), fq))
        out.append([y, g, gg, d.primal, d.tangent, torch.func.vmap(lambda t: f(t, fq))(x.detach().view(2, 3)),
                    torch.func.vmap(torch.func.grad(values(f, fq)))(x.detach().view(2, 3)),
                    torch.func.hessian(values(f, fq))(x.detach().float())])
    for a, b in zip(*out):
        assert a.dtype == b.dtype and torch.equal(a, b)


def test_ste_special_values():
    x = torch.tensor([float("inf"), -float("inf"), float("nan"), 3e38, -1e-45, -0.0, 2.0])
    for fq in (lambda t: torch.ones_like(t), lambda t: t * 0.5):
        assert np.array_equal(ste(x, fq).numpy(), plain(x, fq).numpy(), equal_nan=True)
    assert ste(x[:0], torch.round).shape == (0,)


def test_ste_traced():
    f = torch.compile(lambda t: ste(t, torch.round), backend="eager", fullgraph=True)
    x = torch.tensor([0.4, 1.6], requires_grad=True)
    f(x).sum().backward()
    assert torch.equal(f(x), torch.tensor([0.0, 2.0])) and torch.equal(x.grad, torch.ones(2))
    t = torch.jit.trace(lambda t: ste(t, torch.round), (torch.zeros(2),))
    assert torch.equal(t(torch.tensor([1.4, 2.6])), torch.tensor([1.0, 3.0])) and "PythonOp" not in str(t.graph)
    g, = torch.autograd.grad(ste(x, torch.round), x, torch.eye(2), is_grads_batched=True)
    assert torch.equal(g, torch.eye(2))
