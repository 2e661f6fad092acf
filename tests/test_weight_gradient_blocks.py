"""Weight gradients at every block shape of the kernel (columns below, at and past
a tile; row counts that end inside a step and leave slabs empty) for fp32 and fp16
operands, against float64: at most N additions of products exact to 2^-23."""
import pytest
import torch

from exact_amd.cpp_extension import backward_func as bf


@pytest.mark.gpu
@pytest.mark.parametrize("K,D", [(1, 5), (20, 100), (32, 129), (33, 128), (47, 300), (64, 130), (65, 30), (100, 64), (129, 65), (256, 200)])
@pytest.mark.parametrize("N", [16384, 17003, 70001])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_against_float64(cuda, K, D, N, dtype):
    g = torch.Generator(device=cuda).manual_seed(N + K + D)
    dy = torch.randn(N, K + 3, generator=g, device=cuda).to(dtype)[:, :K]      # a row stride of its own
    x = torch.randn(N, D, generator=g, device=cuda).to(dtype)
    got = bf.weight_gradient(dy, x)
    want, total = dy.double().t() @ x.double(), dy.double().abs().t() @ x.double().abs()
    # sums of at most 512 + 137 rows per slab in fp32, slabs met one by one; one rounding to fp16 at the end
    bound = (6 * 649 + 137) * 2.0 ** -24 * total + (2.0 ** -11 * want.abs() + 2.0 ** -24 if dtype == torch.float16 else 0)
    assert got.dtype == dtype and got.shape == (K, D) and ((got.double() - want).abs() <= bound).all()
