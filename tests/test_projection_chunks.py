"""The projection kernels at the edges of their 64-feature chunks, 16-feature
steps, 4-feature pieces, column tiles and row tiles, on any matrix and on a sign
matrix, with and without the quantiser.  A sum of D fp32 products of which each
is three or six bf16 products in fp32 is wrong by at most 2^-24 of the absolute
terms per addition, 6 D of them, and one rounding per term for what is left out."""
import pytest
import torch

from exact_amd import ops
from exact_amd.conf import config
from exact_amd.cpp_extension import quantization as extq


@pytest.mark.parametrize("signs", [False, True])
@pytest.mark.parametrize("k", [7, 40, 76, 128])                        # one to four column tiles
@pytest.mark.parametrize("N,D", [(1, 1), (33, 3), (31, 4), (32, 5), (65, 63), (40, 64), (33, 65), (32, 66), (1, 67), (64, 127),
                                 (33, 128), (31, 129), (70, 130), (2, 131), (33, 133), (32, 197), (5, 258)])
def test_projection(backend, N, D, k, signs):
    g = torch.Generator().manual_seed(1000 * N + D + k)
    x = torch.randn(N, D, generator=g).to(backend)
    matrix = (2.0 * torch.randint(2, (D, k), generator=g) - 1) / k ** 0.5 if signs else torch.randn(D, k, generator=g)
    matrix = matrix.to(backend)
    if signs:
        matrix._exact_sign_matrix = True

    def source(*_):
        return matrix
    config.rp_matrix_source = source
    reduced, used = ops.input2rp(x, k)
    want = x.double() @ matrix.double()
    bound = (7 * D + 2) * 2.0 ** -24 * (x.double().abs() @ matrix.double().abs()) + 1e-30
    assert reduced.shape == (N, k) and ((reduced.double() - want).abs() <= bound).all()
    # the fused launch quantises exactly these sums
    config.noise_source = lambda shape, device: torch.full(shape, 0.25).to(device)
    for one, two in zip(extq.rp_minmax_pack(x, used, 2), extq.minmax_pack(reduced, 2)):
        assert torch.equal(one, two)


@pytest.mark.parametrize("N,D,k", [(8192, 130, 5), (8200, 131, 33), (8223, 290, 64), (8193, 385, 20), (8200, 639, 80),
                                   (16500, 602, 76)])                    # the last: a second tile for some workgroups
def test_back_by_whole_rows(backend, N, D, k):
    """rp2input of a sign matrix where a workgroup owns whole rows: tiles of 32 rows, steps of 16 features, pieces of four columns."""
    g = torch.Generator().manual_seed(N + D + k)
    matrix = ((2.0 * torch.randint(2, (D, k), generator=g) - 1) / k ** 0.5).to(backend)
    matrix._exact_sign_matrix = True
    x = torch.randn(N, k, generator=g).to(backend)
    got, want = ops.rp2input(x, (N, D), matrix), x.double() @ matrix.double().t()
    bound = (4 * k + 2) * 2.0 ** -24 * (x.double().abs() @ matrix.double().t().abs()) + 1e-30
    assert got.shape == (N, D) and ((got.double() - want).abs() <= bound).all()


@pytest.mark.parametrize("D,k", [(1, 1), (5, 3), (64, 8), (100, 25), (602, 76), (33, 128)])
def test_drawn_matrix(backend, D, k):
    """The matrix and its fragments in one launch: the values of the reference's expression, the fragments of the matrix."""
    draws = torch.randint(2, (D, k), generator=torch.Generator().manual_seed(D), dtype=torch.float32).to(backend)
    got, want = extq.sign_matrix(draws), (2.0 * draws - 1) / k ** 0.5
    assert torch.equal(got, want) and got._exact_sign_matrix
    want._exact_sign_matrix = True
    assert torch.equal(extq.rp_table(got, extq.RP_BF16_SIGNS), extq.rp_table(want, extq.RP_BF16_SIGNS))
    got += 0.0                                                            # written to: the kept table is not used any more
    assert torch.equal(extq.rp_table(got, extq.RP_BF16_SIGNS), extq.rp_table(want, extq.RP_BF16_SIGNS))


def test_drawn_matrix_of_every_width(backend):
    """Bit for bit the framework's (2 b - 1) / sqrt(k) on the device, which multiplies by 1 / sqrt(k) formed in fp64 and
    rounded once; rounding sqrt(k) to fp32 first gives the neighbouring number for 31 of the 128 widths."""
    for k in range(1, extq.RP_PACK_MAX_COLUMNS + 1):
        draws = torch.randint(2, (3, k), dtype=torch.float32).to(backend)
        got = extq.sign_matrix(draws)
        assert torch.equal(got, (2.0 * draws - 1) * torch.tensor(1.0 / k ** 0.5, device=backend)), k
        if backend.type == "cuda":
            assert torch.equal(got, (2.0 * draws - 1) / k ** 0.5), k


def test_drawn_matrices_under_vmap(backend):
    """A draw inside a function transform has no memory of its own: the framework's expression."""
    torch.manual_seed(3)
    got = torch.vmap(lambda x: ops._projection_matrix(12, 5, x.device, x.dtype), randomness="different")(torch.zeros(2, 3, device=backend))
    assert got.shape == (2, 12, 5) and torch.equal(got.abs(), torch.full_like(got, 1.0 / 5 ** 0.5))


def test_drawn_matrices_inside_a_compiled_region(backend):
    """The framework's expression, without a break in the graph."""
    compiled = torch.compile(lambda x: ops._projection_matrix(12, 5, x.device, x.dtype) * 1, backend="eager", fullgraph=True)
    got = compiled(torch.zeros(2, 3, device=backend))
    assert got.shape == (12, 5) and torch.equal(got.abs(), torch.full_like(got, 1.0 / 5 ** 0.5))
