"""Dense products at the ends of the fp32 range: infinities and NaN where fp32
arithmetic puts them, full accuracy for operands that are very large or very
small throughout (a row of X, a column of the matrix, everything)."""
import pytest
import torch

from exact_amd.conf import config
from exact_amd.cpp_extension import backward_func as bf


def _check(x, w, transposed=False, bias=None, addend=None):
    """Against float64: the same infinities and NaN, else within the rounding of an fp32 sum of D terms, each at most
    2^-24 of the sum of the magnitudes, and of the fp32 result itself (2^-149 where that is subnormal)."""
    config.tall_gemm_min_rows = 1
    m = w.double().t() if transposed else w.double()
    want = x.double() @ m
    total = x.double().abs() @ m.abs()
    for extra in (bias, addend):
        if extra is not None:
            want, total = want + extra.double(), total + extra.double().abs()
    into = addend.clone() if addend is not None else None
    got = bf.tall_matmul(x, w, transposed=transposed, bias=bias, addend=into, into=into)
    if bias is None and addend is None:
        assert hasattr(w, "_exact_gemm_table")
    expected = want.float()                                  # infinite where the fp32 range ends
    finite = torch.isfinite(expected)
    assert torch.equal(torch.isnan(got), torch.isnan(expected))
    assert torch.equal(got[~finite & ~torch.isnan(expected)], expected[~finite & ~torch.isnan(expected)])
    bound = (7 * x.shape[1] + 4) * 2.0 ** -24 * total + 2.0 ** -148
    assert ((got.double() - want).abs() <= bound)[finite].all()


def _operands(backend, N, D, K, seed=0):
    g = torch.Generator().manual_seed(1000 * N + 10 * D + K + seed)
    return torch.randn(N, D, generator=g).to(backend), torch.randn(D, K, generator=g).to(backend)


def _rows(w):
    """The matrix as F.linear holds it, [K, D] with a row stride of D."""
    return torch.empty(w.shape[1], w.shape[0], device=w.device).copy_(w.t())


SHAPES = [(40, 18, 1), (33, 34, 40), (131, 6, 96), (70, 66, 130), (64, 32, 256)]     # every number of column tiles per slab


@pytest.mark.parametrize("N,D,K", SHAPES)
def test_infinities_and_nan(backend, N, D, K):
    inf, nan = float("inf"), float("nan")
    x, w = _operands(backend, N, D, K)
    x[0, 0], x[1, 1], x[2, 0], x[2, 1], x[N - 1, D - 1] = inf, -inf, inf, -inf, nan
    _check(x, w)
    w[:, K // 2] = 0.0                                       # infinity times zero
    _check(x, w)
    x, w = _operands(backend, N, D, K, 1)
    w[D - 1, 0], w[0, K - 1] = -inf, nan
    _check(x, w)
    w[0, K - 1] = inf
    x[3] = 0.0
    _check(x, w, bias=torch.ones(K, device=x.device), addend=torch.ones(N, K, device=x.device))
    _check(x, _rows(w), transposed=True)


@pytest.mark.parametrize("N,D,K", SHAPES)
@pytest.mark.parametrize("xs,ws", [(3e-38, 1.0), (1.0, 3e-38), (1e-42, 1.0), (1e-38, 1e30), (1e30, 1e-38), (1e-42, 3e37),
                                   (3e37, 1e-42), (1e-20, 1e-18), (1e-25, 1e-25), (1e38, 1e-3), (1e-3, 1e38), (3e37, 3e37)])
def test_operands_that_are_small_or_large_throughout(backend, N, D, K, xs, ws):
    x, w = _operands(backend, N, D, K)
    _check(x * xs, w * ws)


@pytest.mark.parametrize("N,D,K", SHAPES)
def test_rows_and_columns_of_every_size(backend, N, D, K):
    """Ordinary rows and columns beside rows and columns at the ends of the range, in the same tile."""
    x, w = _operands(backend, N, D, K)
    scale = torch.tensor([1.0, 1e-38, 1e-42, 1e37, 0.0, 1e-30]).to(x.device)
    x = x * scale[torch.arange(N, device=x.device) % 6][:, None]
    w = w * scale[torch.arange(K, device=x.device) % 5][None, :]
    add = torch.randn(N, K, device=x.device)
    _check(x, w)
    _check(x, w, addend=add)
    _check(x, w, bias=add[0].contiguous(), addend=add)


@pytest.mark.parametrize("N,D,K", SHAPES)
def test_the_largest_finite_values(backend, N, D, K):
    """Above bf16's largest number, where rounding to bf16 is infinite."""
    top = torch.finfo(torch.float32).max
    x, w = _operands(backend, N, D, K)
    x[::3, 0], x[1::3, D // 2] = top, -top
    _check(x, w * 0.01)
    x, w = _operands(backend, N, D, K, 1)
    w[0, ::2], w[1, 0] = top, -top
    _check(x * 0.01, w)
    _check(x * 0.01, _rows(w), transposed=True)
