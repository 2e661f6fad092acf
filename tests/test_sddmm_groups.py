"""exact_sddmm_f32 at every lane-group width and its edges (columns below, at and
past a group, no multiple of four, more than one pass), entry counts that end
inside a group, runs that share a row and runs that do not: against float64."""
import pytest
import torch

from exact_amd.cpp_extension import spmm


@pytest.mark.parametrize("K", [1, 3, 4, 5, 31, 32, 33, 64, 65, 128, 130, 256, 259])
@pytest.mark.parametrize("reduce,idx", [("sum", torch.long), ("mean", torch.int32)])
def test_edge_gradients(backend, K, reduce, idx):
    g = torch.Generator().manual_seed(K)
    lengths = torch.tensor([0, 40, 1, 1, 3, 0, 8, 16, 7, 0, 2, 25])
    rowptr = torch.zeros(13, dtype=torch.long)
    rowptr[1:] = lengths.cumsum(0)
    row = torch.repeat_interleave(torch.arange(12), lengths)
    col = torch.randint(0, 19, (row.numel(),), generator=g)
    mat, grad = torch.randn(19, K, generator=g), torch.randn(12, K, generator=g)
    mat[3, K - 1] = float("inf")                       # reaches only the entries of column 3
    got = spmm.spmm_value_bw(row.to(idx).to(backend), rowptr.to(idx).to(backend), col.to(idx).to(backend), mat.to(backend),
                             grad.to(backend), reduce).cpu().double()
    terms = mat.double()[col] * grad.double()[row]
    scale = lengths.double()[row] if reduce == "mean" else torch.ones(row.numel(), dtype=torch.double)
    want, finite = terms.sum(1) / scale, col != 3
    assert torch.equal(got[~finite], want[~finite])    # +-inf with grad's sign
    bound = (K + 2) * 2.0 ** -24 * terms.abs().sum(1) / scale
    assert ((got - want).abs()[finite] <= bound[finite]).all()
