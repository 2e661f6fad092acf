"""A GraphSAGE layer in evaluation mode without gradients (the narrow side of
lin_l aggregated, tall GEMMs) against the same layer with gradients enabled,
which runs the separate operations."""
import pytest
import torch

import exact_amd as exact
from exact_amd.sparse import SparseTensor


@pytest.mark.gpu
@pytest.mark.parametrize("cin,cout,bias", [(48, 20, True), (20, 48, True), (33, 33, False)])
@pytest.mark.parametrize("N", [500, 17000])           # below and above the rows from which the library's GEMM runs
@pytest.mark.parametrize("valued", [False, True])
def test_same_as_the_separate_operations(cuda, cin, cout, bias, N, valued):
    g = torch.Generator().manual_seed(N + cin)
    src, dst = torch.randint(0, N, (6 * N,), generator=g), torch.randint(0, N // 2, (6 * N,), generator=g)
    value = torch.rand(6 * N, generator=g).to(cuda) if valued else None
    adj = SparseTensor.from_edge_index(dst.to(cuda), src.to(cuda), value, (N, N))
    layer = exact.QSAGEConv(cin, cout, bias=bias).to(cuda).eval()
    x = torch.randn(N, cin, generator=g).to(cuda)
    want = layer(x, adj).detach()
    with torch.no_grad():
        got = layer(x, adj)
    # two fp32 sums of `cin` terms in another order, of values of order one
    assert (got - want).abs().max() <= 4 * cin * 2.0 ** -24 * max(1.0, want.abs().max().item())
    with torch.no_grad():                              # an input that is read twice is not written
        again = layer(x, adj)
    assert (again - got).abs().max() <= 4 * cin * 2.0 ** -24 * max(1.0, want.abs().max().item())
    with torch.no_grad():                              # a fp64 input takes the general path, and fails as it did
        with pytest.raises(RuntimeError):
            layer(x.double(), adj)
