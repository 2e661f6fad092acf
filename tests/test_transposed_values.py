"""The transposed operands of learned edge values: gathered values against the
framework's gather, and the kept row indices never older than their tensors."""
import pytest
import torch

from exact_amd.cpp_extension import spmm


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("index", [torch.int32, torch.int64])
@pytest.mark.parametrize("n", [1, 255, 2048, 2049, 5000])              # below, at and past a workgroup's 2048 entries
def test_gather(backend, n, index, dtype):
    g = torch.Generator().manual_seed(n)
    value = torch.randn(n, generator=g).to(dtype)
    value[0], value[n // 2] = float("inf"), float("nan")
    order = torch.randperm(n, generator=g)
    got = spmm._transposed_values(value.to(backend), order.to(index).to(backend))
    assert got.dtype == torch.float32
    assert torch.equal(torch.nan_to_num(got.cpu(), nan=7.5), torch.nan_to_num(value.float()[order], nan=7.5))


def test_strided_values_take_the_frameworks_gather(backend):
    value = torch.arange(12.0).to(backend)[::3]
    assert torch.equal(spmm._transposed_values(value, torch.tensor([2, 0, 3]).to(backend)).cpu(), torch.tensor([6.0, 0.0, 9.0]))


def test_values_that_do_not_lie_in_plain_memory_take_the_frameworks_gather(backend):
    value, order = torch.arange(3.0).to(backend), torch.tensor([2, 0, 1]).to(backend)
    want = value[order]
    assert torch.equal(spmm._transposed_values(torch._neg_view(value), order), -want)
    assert torch.equal(torch.vmap(spmm._transposed_values, (0, None))(torch.stack([value, 2 * value]), order), torch.stack([want, 2 * want]))


def test_rows_follow_their_tensors(backend):
    row, order = torch.tensor([0, 0, 1, 2]).to(backend), torch.tensor([1, 3, 0, 2]).to(backend)
    first = spmm._transposed_rows(row, order)
    assert torch.equal(first, row[order])
    row[3] = 1                                              # in place
    assert torch.equal(spmm._transposed_rows(row, order), row[order])
    order.copy_(torch.tensor([3, 2, 1, 0]))
    assert torch.equal(spmm._transposed_rows(row, order), row[order])
    other = torch.tensor([2, 1, 0, 0]).to(backend)          # other rows with the same permutation
    assert torch.equal(spmm._transposed_rows(other, order), other[order])
    kept = len(spmm._ROW_CSC)
    del order
    assert len(spmm._ROW_CSC) < max(kept, 1) or kept == 0   # gone with the permutation
    with torch.inference_mode():
        frozen = torch.tensor([1, 0]).to(backend)
    assert torch.equal(spmm._transposed_rows(torch.tensor([4, 5]).to(backend), frozen).cpu(), torch.tensor([5, 4]))


@pytest.mark.gpu
def test_rows_under_capture_and_on_another_stream(cuda):
    row, order = torch.randint(9, (50,), device=cuda), torch.randperm(50, device=cuda)
    want = row[order]
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        assert torch.equal(spmm._transposed_rows(row, order), want)
        graph = torch.cuda.CUDAGraph()
        torch.cuda.synchronize()
        with torch.cuda.graph(graph, stream=side):
            captured = spmm._transposed_rows(row, order)
    torch.cuda.synchronize()
    row.zero_()
    graph.replay()
    torch.cuda.synchronize()
    assert not captured.any()                               # the replay gathers the rows of its time
    assert torch.equal(spmm._transposed_rows(row, order), row[order])
