"""Which routine takes a call, where the line follows from measurements of both:
below it the framework's routine (or the widened operand) runs as it did."""
import pytest
import torch

from exact_amd import _lib, ops
from exact_amd.cpp_extension import spmm


@pytest.fixture
def calls(backend, monkeypatch):
    """The entry points that are asked for, in order, and the device."""
    real, seen = _lib.lib(), []

    class Spy:
        def __getattr__(self, name):
            seen.append(name)
            return getattr(real, name)
    monkeypatch.setattr(_lib, "lib", lambda: Spy())
    return seen, backend


@pytest.mark.parametrize("K,shift,direct", [(8, 0, False), (64, 0, False), (66, 0, True), (101, 0, False), (128, 0, True), (128, 1, False), (128, 2, True)])
def test_half_operands_of_the_sparse_product(calls, K, shift, direct):
    """As they are from 66 even columns on a 4-byte boundary on, widened otherwise; the same product either way."""
    seen, device = calls
    g = torch.Generator().manual_seed(K)
    n = 50
    row = torch.randint(0, n, (400,), generator=g).sort().values
    col = torch.randint(0, n, (400,), generator=g)
    rowptr = torch.zeros(n + 1, dtype=torch.long)
    rowptr[1:] = torch.bincount(row, minlength=n).cumsum(0)
    wide = torch.randn(n, K + 4, generator=g).half().to(device)
    mat = wide[:, shift:shift + K]
    got = spmm.spmm_csr(rowptr.to(device), col.to(device), None, mat, "sum")
    assert ("exact_spmm_csr_strided_f16" in seen) == direct and ("exact_spmm_csr_strided_f32" in seen) == (not direct)
    want = torch.zeros(n, K, dtype=torch.double).index_add_(0, row, mat.cpu().double()[col])
    assert got.dtype == torch.float16 and ((got.cpu().double() - want).abs() <= 2.0 ** -11 * want.abs() + 1e-4).all()


@pytest.mark.parametrize("N,K,own", [(1024, 16, False), (8000, 8, False), (8192, 8, True)])
def test_statistics_of_a_batch_norm_layer(calls, N, K, own):
    seen, device = calls
    x = (torch.randn(N, K) + 2).to(device).requires_grad_()
    rm, rv, w, b = (t.to(device) for t in (torch.zeros(K), torch.ones(K), torch.ones(K), torch.zeros(K)))
    y = ops.qbatch_norm.apply(x, rm, rv, w, b, True, 0.1, 1e-5, None)
    assert ("exact_bn_statistics_f32" in seen) == own
    want = (x.detach().double() - x.detach().double().mean(0)) / (x.detach().double().var(0, unbiased=False) + 1e-5).sqrt()
    assert (y.detach().double() - want).abs().max() < 1e-4
    y.backward(torch.ones_like(y))
