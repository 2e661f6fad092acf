"""A backward that is itself recorded (create_graph): the batch norm's and the
fp16 weight gradient's stay differentiable where the framework's routines are."""
import pytest
import torch

from exact_amd import ops
from exact_amd.cpp_extension import backward_func as bf


@pytest.mark.parametrize("N,K", [(1200, 300), (1500, 8)])      # below 4096 rows: the framework's backward, which has one of its own
def test_batch_norm(backend, N, K):
    g = torch.Generator().manual_seed(N)
    x = torch.randn(N, K, generator=g).to(backend).requires_grad_()
    w, b = (torch.rand(K, generator=g) + 0.5).to(backend).requires_grad_(), torch.zeros(K).to(backend).requires_grad_()
    rm, rv = torch.zeros(K).to(backend), torch.ones(K).to(backend)
    dy = torch.randn(N, K, generator=g).to(backend).requires_grad_()
    y = ops.qbatch_norm.apply(x, rm, rv, w, b, True, 0.1, 1e-5, None)
    dx, dw, db = torch.autograd.grad(y, (x, w, b), dy, create_graph=True)
    assert dx.requires_grad and dw.requires_grad and db.requires_grad
    second = torch.autograd.grad(dx.square().sum() + dw.square().sum() + db.square().sum(), (dy, w))
    assert all(torch.isfinite(t).all() and t.abs().max() > 0 for t in second)
    # d(db^2)/d(dy) alone: 2 db on every row
    y = ops.qbatch_norm.apply(x, rm, rv, w, b, True, 0.1, 1e-5, None)
    db, = torch.autograd.grad(y, b, dy, create_graph=True)
    per_row, = torch.autograd.grad(db.square().sum(), dy)
    assert torch.allclose(per_row, (2 * dy.detach().sum(0)).expand(N, K), rtol=1e-4, atol=1e-4)


def test_half_weight_gradient(backend):
    g = torch.Generator().manual_seed(3)
    dy = torch.randn(16400, 4, generator=g).half().to(backend).requires_grad_()
    x = torch.randn(16400, 6, generator=g).half().to(backend)
    out = bf.weight_gradient(dy, x)
    assert out.requires_grad
    back, = torch.autograd.grad(out.float().sum(), dy)
    assert torch.allclose(back.float(), x.float().sum(1, keepdim=True).expand(-1, 4), rtol=1e-2, atol=1e-2)
    with torch.no_grad():
        assert not bf.weight_gradient(dy, x).requires_grad
