"""exact_tall_product_f32 at the edges of its column slabs, k-steps and row
blocks, with every epilogue, and exact_rp_bwd_bf16_f32 at row widths that are no
multiple of four: against float64.  An element is the sum of six bf16 products
per feature in fp32, in whatever order the accumulator takes them: at most
6 D + 2 additions (the bias and the addend among them), each wrong by at most
2^-24 of the sum of the absolute terms, and the products left out are below one
such rounding per feature."""
import pytest
import torch

from exact_amd import ops
from exact_amd.conf import config
from exact_amd.cpp_extension import backward_func as bf


# K: one tile, tiles of one slab, padded slabs (5 = 3 + 2, 9 = 3 x 3, 11 = 4 + 4 + 3 tiles); D: below, at and past a step
@pytest.mark.parametrize("D", [2, 16, 34, 70])
@pytest.mark.parametrize("K", [1, 33, 96, 129, 160, 270, 330])
@pytest.mark.parametrize("N", [31, 160])
def test_tall_product(backend, N, D, K):
    config.tall_gemm_min_rows = 1
    g = torch.Generator().manual_seed(N + 7 * D + 31 * K)
    x = torch.randn(N, D, generator=g).to(backend)
    w = torch.randn(K, D, generator=g).to(backend)
    b, c = torch.randn(K, generator=g).to(backend), torch.randn(N, K + 3, generator=g).to(backend)[:, :K]
    want = x.double() @ w.double().t()
    bound = (7 * D + 2) * 2.0 ** -24 * ((x.abs().double() @ w.abs().double().t()) + b.abs().double() + c.abs().double()) + 1e-30
    assert ((bf.tall_matmul(x, w, transposed=True).double() - want).abs() <= bound).all()
    assert ((bf.tall_matmul(x, w, transposed=True, bias=b).double() - want - b.double()).abs() <= bound).all()
    got = bf.tall_matmul(x, w.t().contiguous(), bias=b, addend=c)
    assert ((got.double() - want - b.double() - c.double()).abs() <= bound).all()
    into = torch.full((N, K + 2), 9.0).to(backend)
    into[:, :K] = c
    bf.tall_matmul(x, w, transposed=True, addend=into[:, :K], into=into[:, :K])
    assert ((into[:, :K].double() - want - c.double()).abs() <= bound).all() and (into[:, K:] == 9.0).all()


@pytest.mark.parametrize("D", [1, 6, 127, 130, 602])
@pytest.mark.parametrize("k", [3, 20, 76])
def test_projection_back_to_any_width(backend, D, k):
    g = torch.Generator().manual_seed(D + k)
    r = torch.randn(D, k, generator=g).to(backend)
    x = torch.randn(261, k, generator=g).to(backend)
    got = ops.rp2input(x, (261, D), r)
    want, bound = x.double() @ r.double().t(), (7 * k + 2) * 2.0 ** -24 * (x.abs().double() @ r.abs().double().t()) + 1e-30
    assert got.shape == (261, D) and ((got.double() - want).abs() <= bound).all()


def test_few_workgroups_and_a_deep_sum_stay_with_the_framework(backend):
    """The sizes rule: 200 rows make two workgroups, which take 160 features and no more; a depth set by hand is obeyed."""
    config.tall_gemm_min_rows = 1
    x = torch.randn(200, 162).to(backend)

    def taken(d, k):
        w = torch.randn(k, d).to(backend)
        bf.tall_matmul(x[:, :d].contiguous(), w, transposed=True)
        return hasattr(w, "_exact_gemm_table")
    assert taken(160, 40) and not taken(162, 40)
    config.tall_gemm_min_depth = 1
    assert taken(162, 40) and taken(162, 100)
    worth = bf._worth_a_tall_product
    assert worth(16384, 128, 256) and not worth(16384, 256, 256) and worth(16384, 4096, 600)
    assert worth(40000, 602, 40) and not worth(40000, 602, 16) and not worth(40000, 1024, 40) and worth(40000, 1024, 256)
    assert worth(169343, 256, 256) and worth(2449029, 100, 256)
