"""Sparse products at the sizes where the split into chunks changes (chunks of 64,
128 and 256 entries; rows in pieces or owned whole), on rows that end at, just
before and just after chunk boundaries, empty rows and hubs, for fp32 and fp16
operands: against float64, within the rounding of a sum of the row's length."""
import pytest
import torch

from exact_amd.cpp_extension import spmm


def _graph(lengths, n_cols, seed):
    g = torch.Generator().manual_seed(seed)
    rowptr = torch.zeros(len(lengths) + 1, dtype=torch.long)
    rowptr[1:] = torch.tensor(lengths).cumsum(0)
    nnz = int(rowptr[-1])
    return rowptr, torch.randint(0, n_cols, (nnz,), generator=g), torch.randn(nnz, generator=g)


def _check(device, lengths, K, dtype, reduce, valued, idx):
    n_cols = 97
    rowptr, col, val = _graph(lengths, n_cols, K + len(lengths))
    x = torch.randn(n_cols, K, generator=torch.Generator().manual_seed(K)).to(dtype)
    val = val if valued else None
    rowptr, col, x, lengths = rowptr.to(device), col.to(device), x.to(device), torch.tensor(lengths, device=device)
    val = None if val is None else val.to(device)
    got = spmm.spmm_csr(rowptr.to(idx), col.to(idx), val, x, reduce)
    row = torch.repeat_interleave(torch.arange(len(lengths), device=device), lengths)
    terms = x.double()[col] * (1.0 if val is None else val.double()[:, None])
    want = torch.zeros(len(lengths), K, dtype=torch.double, device=device).index_add_(0, row, terms)
    total = torch.zeros(len(lengths), K, dtype=torch.double, device=device).index_add_(0, row, terms.abs())
    count = lengths.double().clamp(min=1)[:, None]
    if reduce == "mean":
        want, total = want / count, total / count
    # pieces of at most 64 serial additions, then the pieces; one more rounding to fp16
    bound = (64 + count / 64 + 4) * 2.0 ** -24 * total + (2.0 ** -11 * want.abs() + 2.0 ** -24 if dtype == torch.float16 else 0)
    assert got.dtype == dtype and ((got.double() - want).abs() <= bound).all()


EDGES = [0, 64, 63, 1, 65, 0, 0, 128, 127, 129, 1, 0, 256, 255, 257, 2, 62, 64, 64, 3000, 0, 5, 520, 0]


@pytest.mark.parametrize("K,dtype", [(47, torch.float32), (130, torch.float32), (70, torch.float16), (132, torch.float16), (131, torch.float16)])
@pytest.mark.parametrize("reduce,valued,idx", [("sum", True, torch.int32), ("mean", False, torch.long)])
def test_row_edges(backend, K, dtype, reduce, valued, idx):
    _check(backend, EDGES, K, dtype, reduce, valued, idx)
    _check(backend, [0] * 70 + EDGES[::-1] + [1] * 200 + [0] * 300 + [1, 0] * 40, K, dtype, reduce, valued, idx)


@pytest.mark.gpu
@pytest.mark.parametrize("copies,K,dtype", [(90, 20, torch.float32), (450, 20, torch.float32), (3400, 20, torch.float32),   # one element per lane
                                            (60, 130, torch.float32), (120, 130, torch.float32), (300, 130, torch.float32),
                                            (1700, 130, torch.float32),                                              # two
                                            (60, 132, torch.float16), (300, 132, torch.float16), (3400, 132, torch.float16)])   # four
def test_every_split(cuda, copies, K, dtype):
    for reduce, valued, idx in (("sum", True, torch.int32), ("mean", False, torch.long)):
        _check(cuda, EDGES * copies, K, dtype, reduce, valued, idx)
