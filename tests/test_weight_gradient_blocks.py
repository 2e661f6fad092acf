"""Weight gradients at every block shape of the kernels (columns below, at and past
a tile; row counts that end inside a step and leave slabs empty) for fp32 and fp16
operands.  Sparse integers, whose sums are exact whatever the order, have to give
the float64 product bit for bit: a row lost or counted twice shows, and so does a
piece of an operand, as the integers use every bit of it.  Dense random operands
have to stay within what the rounding of fp32 sums can do."""
import pytest
import torch

from exact_amd import layers
from exact_amd.conf import config
from exact_amd.cpp_extension import backward_func as bf

SHAPES = [(1, 5), (20, 100), (32, 129), (33, 128), (47, 300), (64, 130), (65, 30), (100, 64), (129, 65), (256, 200)]
DTYPES = [torch.float32, torch.float16]


def _sparse_integers(N, K, D, dtype, device):
    """dy holds 1, -1 or 2 in about eight rows a column, the last row among them, x integers of 20 (fp32) or 11 bits:
    sums below 2^24 in fp32, below 2^16 in fp16."""
    g = torch.Generator().manual_seed(N + K + D)
    dy = torch.zeros(N, K)
    rows = torch.cat([torch.randint(0, N, (6, K), generator=g), torch.full((1, K), N - 1), torch.zeros(1, K, dtype=torch.long)])
    dy.scatter_(0, rows, torch.tensor([1.0, -1.0, 2.0])[torch.randint(0, 3, (8, K), generator=g)])
    top = 2 ** 20 if dtype == torch.float32 else 2 ** 11
    x = torch.randint(-top + 1, top, (N, D), generator=g).float()
    return dy.to(device, dtype), x.to(device, dtype)


def _check_integers(device, N, K, D, dtype):
    dy, x = _sparse_integers(N, K, D, dtype, device)
    want = (dy.double().t() @ x.double()).to(dtype)                      # one rounding to fp16
    got = bf.weight_gradient(dy, x)
    assert got.dtype == dtype and torch.equal(got, want)
    wide_dy = torch.full((N, K + 3), float("nan"), dtype=dtype, device=device)   # row strides of their own, NaN between
    wide_x = torch.full((N, D + 5), float("nan"), dtype=dtype, device=device)
    wide_dy[:, 1:1 + K], wide_x[:, 3:3 + D] = dy, x
    assert torch.equal(bf.weight_gradient(wide_dy[:, 1:1 + K], wide_x[:, 3:3 + D]), want)


@pytest.mark.gpu
@pytest.mark.parametrize("K,D", SHAPES)
@pytest.mark.parametrize("N", [16384, 17003, 70001])
@pytest.mark.parametrize("dtype", DTYPES)
def test_integers_are_exact(cuda, K, D, N, dtype):
    _check_integers(cuda, N, K, D, dtype)


@pytest.mark.parametrize("K,D", [(20, 40), (33, 33)])
@pytest.mark.parametrize("dtype", DTYPES)
def test_integers_are_exact_on_the_emulated_kernels(backend, K, D, dtype):
    _check_integers(backend, 16397, K, D, dtype)


@pytest.mark.gpu
@pytest.mark.parametrize("K,D", SHAPES)
@pytest.mark.parametrize("N", [16384, 17003, 70001])
@pytest.mark.parametrize("dtype", DTYPES)
def test_against_float64(cuda, K, D, N, dtype):
    g = torch.Generator(device=cuda).manual_seed(N + K + D)
    dy = torch.randn(N, K + 3, generator=g, device=cuda).to(dtype)[:, :K]      # a row stride of its own
    x = torch.randn(N, D, generator=g, device=cuda).to(dtype)
    got = bf.weight_gradient(dy, x)
    want = dy.double().t() @ x.double()
    # A slab sums up to 700 products one after the other; with terms of random sign its rounding errors, 0.3 x 2^-24 of
    # a running sum that grows as the square root, come to 0.3 x sqrt(700 / 2) x 2^-24 of the slab's rms, and slabs add
    # in squares: a standard deviation of 6 x 2^-24 of the rms of the whole.  Ten of them; an operand that lost all but
    # one bf16 piece is off by 2^-10 of the rms, two hundred times this.
    rms = ((dy.double() ** 2).t() @ (x.double() ** 2)).sqrt()
    bound = 60 * 2.0 ** -24 * rms + (2.0 ** -11 * want.abs() + 2.0 ** -25 if dtype == torch.float16 else 0)
    assert got.dtype == dtype and got.shape == (K, D) and ((got.double() - want).abs() <= bound).all()


@pytest.mark.parametrize("K,D", [(20, 40), (70, 35)])
def test_half_operands_at_the_ends_of_their_range(backend, K, D):
    """Infinities and NaN where fp32 sums put them, subnormal fp16 numbers kept, sums past 65504 infinite."""
    N, inf = 16397, float("inf")
    dy, x = _sparse_integers(N, K, D, torch.float16, backend)
    dy[:, 3] *= 2.0 ** -24                                               # subnormal: 1, 2 units of the last place
    dy[100, 4], dy[N - 1, 5] = 1000.0, float("nan")
    dy[200, 6], dy[201, 6] = inf, -inf
    x[100, 0], x[200, 1], x[201, 1] = 600.0, 2.0, 2.0
    x[N - 1, 7] = inf                                                    # times dy[N - 1] != 0
    want = (dy.double().t() @ x.double()).half()
    got = bf.weight_gradient(dy, x)
    assert torch.isinf(want).any() and torch.isnan(want).any() and (want[3].double() != 0).any()
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(got.nan_to_num(7.0, 8e4, -8e4), want.nan_to_num(7.0, 8e4, -8e4))


@pytest.mark.parametrize("K,D", [(20, 40), (70, 35)])
def test_half_operands_give_equal_bits_twice(backend, K, D):
    g = torch.Generator().manual_seed(5)
    dy, x = torch.randn(16500, K, generator=g).half().to(backend), torch.randn(16500, D, generator=g).half().to(backend)
    first = bf.weight_gradient(dy, x)
    for _ in range(3):
        assert torch.equal(bf.weight_gradient(dy, x), first)


# one, several and partial blocks; N: the shortest, whole slabs of 64, a last slab of one row
@pytest.mark.parametrize("K,D", [(1, 1), (33, 128), (32, 130), (64, 70), (40, 256), (130, 32), (96, 64), (65, 100), (256, 256)])
@pytest.mark.parametrize("N", [4096, 4161, 5000])
def test_short_batches(backend, N, K, D):
    """In a fixed order, infinities where fp32 has them, and off by what the rounding of the sums does: a slab adds some 64 to
    80 rows one after the other (a standard deviation of 0.3 x sqrt(80 / 2) x 2^-24 of its rms), about ten slabs follow each
    other in eight chains (0.3 x sqrt(10 / 2) of the whole) and the chains are added (0.3 x sqrt(8 / 2)): 2.2 x 2^-24 of the
    rms of the whole, and ten of them are allowed.  An operand cut to 16 bits is off by 2^-17 of the rms, 128 x 2^-24."""
    if N > 4096 and K * D > 20000 and backend.type == "cpu":
        pytest.skip("slow on the emulator")
    g = torch.Generator().manual_seed(N + 7 * K + D)
    dy = torch.randn(N, K + 2, generator=g)[:, :K].to(backend)
    x = torch.randn(N, D, generator=g).to(backend)
    calls = []
    real = bf._scratch_size
    bf._scratch_size = lambda *a: calls.append(a[0]) or real(*a)
    try:
        got = bf.weight_gradient(dy, x)
        again = bf.weight_gradient(dy, x)
        dy[3, 0], x[N - 1, D - 1] = float("inf"), float("-inf")
        ends = bf.weight_gradient(dy, x)
    finally:
        bf._scratch_size = real
    assert calls == ["exact_linear_dw_short_work_nbytes"] * 3 and torch.equal(got, again)
    dy[3, 0] = x[N - 1, D - 1] = 0.0
    # (both tensors had a finite value there before: compare what those rows do not reach)
    want, bound = dy.double().t() @ x.double(), 22 * 2.0 ** -24 * ((dy.double() ** 2).t() @ (x.double() ** 2)).sqrt()
    keep = torch.ones(K, D, dtype=torch.bool, device=got.device)
    keep[0, :] = False
    keep[:, D - 1] = False
    assert ((got.double() - want).abs() <= bound)[keep].all()
    if K > 1 and D > 1:
        assert torch.isinf(ends[0, : D - 1]).all() and torch.isinf(ends[1:, D - 1]).all()
        assert torch.equal(ends[1:, : D - 1], got[1:, : D - 1])


@pytest.mark.parametrize("K,D", [(1, 5), (20, 40), (33, 128), (65, 100), (130, 32)])
@pytest.mark.parametrize("N", [4096, 4161])
def test_integers_are_exact_in_short_batches(backend, N, K, D):
    _check_integers(backend, N, K, D, torch.float32)


def test_short_batches_under_a_recorded_backward(backend):
    dy, x = torch.randn(4096, 3).to(backend).requires_grad_(), torch.randn(4096, 5).to(backend)
    out = bf.weight_gradient(dy, x)
    back, = torch.autograd.grad(out.sum(), dy)
    assert torch.allclose(back, x.sum(1, keepdim=True).expand(-1, 3), atol=1e-4)


@pytest.mark.parametrize("N", [4096, 5000])
def test_short_batches_whose_values_do_not_lie_in_plain_memory(backend, N):
    """Function transforms, batched backward passes, sparse layouts and negated views: the framework's product, as
    outside the range of the kernel."""
    g = torch.Generator().manual_seed(N)
    dy, x = torch.randn(3, N, 4, generator=g).to(backend), torch.randn(N, 5, generator=g).to(backend)
    want = torch.stack([one.t().mm(x) for one in dy])
    close = lambda got: torch.allclose(got, want, rtol=1e-4, atol=1e-3)     # noqa: E731  (sums of N products in two orders)
    assert close(torch.vmap(bf.weight_gradient, (0, None))(dy, x))
    assert close(torch.stack([torch.func.functionalize(bf.weight_gradient)(one, x) for one in dy]))
    assert close(torch.stack([bf.weight_gradient(one, x.to_sparse_csr()) for one in dy]))
    assert close(torch.stack([-bf.weight_gradient(torch._neg_view(one), x) for one in dy]))
    layer = layers.QLinear(5, 4, bias=False).to(backend).train()
    config.compress_activation = False
    got, = torch.autograd.grad(layer(x), layer.weight, dy, is_grads_batched=True)
    assert close(got)


def test_short_batches_inside_a_compiled_region(backend):
    """The framework's product, without a break in the graph."""
    g = torch.Generator().manual_seed(2)
    dy, x = torch.randn(4200, 6, generator=g).to(backend), torch.randn(4200, 9, generator=g).to(backend)
    compiled = torch.compile(bf.weight_gradient, backend="eager", fullgraph=True)
    assert torch.equal(compiled(dy, x), dy.t().mm(x))
