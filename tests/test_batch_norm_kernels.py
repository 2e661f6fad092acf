"""The batch norm on wide matrices and on the packed copy of its input
(exact_bn_statistics_f32, exact_bn_apply_f32, exact_bn_backward_ordered_f32) against
the same formulas in float64 on the dequantised input."""
import numpy as np
import pytest
import torch

from exact_amd import _lib, layers, ops
from exact_amd.conf import config
from exact_amd.cpp_extension import _checks
from exact_amd.cpp_extension import backward_func as bf
from exact_amd.cpp_extension import quantization as extq


# a width below, at and above one column block (1024 columns in fours, 256 otherwise); rows that end inside a pass
@pytest.mark.parametrize("N,K", [(1024, 1), (1027, 100), (1500, 257), (2049, 512), (1025, 1028), (1030, 1100)])
def test_statistics_and_normalisation(backend, N, K):
    g = torch.Generator().manual_seed(N + K)
    x = torch.randn(N, K, generator=g) * 1.5 + 40.0          # mean 27 deviations from zero
    w, b = torch.rand(K, generator=g) + 0.5, torch.randn(K, generator=g)
    rm, rv = torch.randn(K, generator=g).to(backend), torch.rand(K, generator=g).to(backend)
    rm0, rv0, versions = rm.cpu().double(), rv.cpu().double(), (rm._version, rv._version)
    mean, invstd, mult = bf.batch_norm_statistics(x.to(backend), w.to(backend), rm, rv, 0.3, 1e-5)
    var64, mean64 = torch.var_mean(x.double(), dim=0, unbiased=False)
    inv64 = torch.rsqrt(var64 + 1e-5)
    # the mean rounds at 40: 2^-24 * 40, a few times; the moments of about one unit carry 1e-6 relative
    assert (mean.cpu() - mean64).abs().max() < 2e-5
    assert ((invstd.cpu() - inv64) / inv64).abs().max() < 1e-5 and ((mult.cpu() - w * inv64) / (w * inv64)).abs().max() < 1e-5
    assert (rm.cpu() - (0.7 * rm0 + 0.3 * mean64)).abs().max() < 1e-5
    assert (rv.cpu() - (0.7 * rv0 + 0.3 * var64 * N / (N - 1))).abs().max() < 1e-4
    assert rm._version > versions[0] and rv._version > versions[1]
    y = bf.batch_norm_apply(x.to(backend), mean, mult, b.to(backend))
    assert (y.cpu() - ((x - mean64) * inv64 * w + b)).abs().max() < 1e-4


@pytest.mark.parametrize("bits", [1, 2, 4, 8])
@pytest.mark.parametrize("N,K,masked", [(1024, 4, True), (1031, 100, True), (1029, 256, False), (1026, 1028, True)])
def test_backward_from_the_packed_input(backend, bits, N, K, masked):
    g = torch.Generator().manual_seed(N + K + bits)
    x = torch.randn(N, K, generator=g).to(backend)
    dy = torch.randn(N, K, generator=g).to(backend)
    w = (torch.rand(K, generator=g) + 0.5).to(backend)
    p = 0.3 if masked else 0.0
    mask = extq.relu_dropout_fwd(torch.randn(N, K, generator=g).to(backend), p)[1] if masked else None
    packed, scale, mn = extq.minmax_pack(x, bits)
    mean, invstd, _ = bf.batch_norm_statistics(x, w, None, None, 0.1, 1e-5)
    dx, dw, db = bf.batch_norm_backward_packed(dy, mask, p, (packed, bits, scale, mn), w, mean, invstd, [True, True, True])
    x_hat = extq.unpack_bf16param(packed, bits, scale, mn, N, K).double()
    gr = (extq.dropout_bwd(dy, mask, p) if masked else dy).double()
    xmu, inv = x_hat - mean.double(), invstd.double()
    s0, s1 = gr.sum(0), (gr * xmu).sum(0)
    want = (gr - s0 / N - xmu * inv * inv * s1 / N) * inv * w.double()
    assert (dx - want).abs().max() < 1e-5 * want.abs().max()
    assert (db - s0).abs().max() < 1e-6 * gr.abs().sum(0).max()
    assert (dw - s1 * inv).abs().max() < 2e-6 * (gr * xmu).abs().sum(0).max()
    only = bf.batch_norm_backward_packed(dy, mask, p, (packed, bits, scale, mn), None, mean, invstd, [False, False, True])
    assert only[0] is None and only[1] is None and (only[2] - s0).abs().max() < 1e-6 * gr.abs().sum(0).max()


def test_what_the_kernels_do_not_take_goes_to_the_separate_routines(backend):
    x, dy = torch.randn(1100, 10).to(backend), torch.randn(1100, 10).to(backend)
    packed, scale, mn = extq.minmax_pack(x, 2)
    mean, invstd, _ = bf.batch_norm_statistics(x, None, None, None, 0.1, 1e-5)
    copy = (packed, 2, scale, mn)
    want = [True, True, True]
    assert bf.batch_norm_backward_packed(dy, None, 0.0, copy, None, mean, invstd, want) is None            # 10 % 4
    assert bf.batch_norm_statistics(x[:, :9], None, None, None, 0.1, 1e-5) is None                         # strided
    assert bf.batch_norm_statistics(x[:1000], None, None, None, 0.1, 1e-5) is None                         # short
    assert bf.batch_norm_statistics(x, None, torch.zeros(9).to(backend), torch.zeros(9).to(backend), 0.1, 1e-5) is None
    config.deterministic_reductions = True
    assert bf.batch_norm_statistics(x, None, None, None, 0.1, 1e-5) is None
    kept = ops.CompressedActivation(copy, None, x.shape, x.shape)
    config.simulate = True
    assert ops._batch_norm_backward_packed(dy, None, 0.0, kept, None, mean, invstd, want) is None


def _rows(kind, N, K, g):
    """Row orders that a sampled centre, or sums that run through the rows, get wrong."""
    x = torch.randn(N, K, generator=g)
    i = torch.arange(N)[:, None].float()
    if kind == "periodic":                                   # every 512th row far off, with the period of N / 256 and of any power of two
        x[::512] += 100.0
    elif kind == "sorted":
        x = (x * 0.01 + torch.linspace(-50.0, 50.0, N)[:, None]).sort(0).values
    elif kind == "first rows":
        x[:N // 64] += 1000.0
    elif kind == "far from zero":
        x = x * 0.01 + 300.0
    elif kind == "alternating":
        x = x * 1e-3 + torch.where(i % 2 == 0, 5.0, -5.0)
    return x.contiguous()


def _check_statistics(backend, kind, N, K):
    g = torch.Generator().manual_seed(N + K)
    x = _rows(kind, N, K, g)
    mean, invstd, _ = bf.batch_norm_statistics(x.to(backend), None, None, None, 0.1, 0.0)
    var64, mean64 = torch.var_mean(x.double(), dim=0, unbiased=False)
    var = 1.0 / invstd.cpu().double() ** 2
    # a few roundings per join, and the rounding of a mean far from zero, squared, is all that the variance can carry
    assert ((var - var64).abs() <= 2e-6 * var64 + (4 * 2.0 ** -24 * mean64.abs()) ** 2).all()
    assert ((mean.cpu() - mean64).abs() <= 4 * 2.0 ** -24 * (mean64.abs() + var64.sqrt())).all()


KINDS = ["plain", "periodic", "sorted", "first rows", "far from zero", "alternating"]


# rows enough for the eight-row loop of every workgroup, in fours and (3 columns) one by one
@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("N,K", [(65536, 8), (30011, 3), (131072, 4)])
def test_statistics_whatever_the_order_of_the_rows(backend, kind, N, K):
    _check_statistics(backend, kind, N, K)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("N,K", [(131072, 256), (262144, 512), (70001, 301), (169343, 1028), (1000000, 16)])
def test_statistics_whatever_the_order_of_the_rows_at_scale(cuda, kind, N, K):
    _check_statistics(cuda, kind, N, K)


def test_statistics_of_equal_rows_and_of_values_at_the_end_of_the_range(backend):
    x = torch.full((5000, 12), 0.1).to(backend)
    mean, invstd, _ = bf.batch_norm_statistics(x, None, None, None, 0.1, 1e-5)
    assert torch.equal(mean, x[0]) and ((invstd - 1e-5 ** -0.5).abs() < 1e-3).all()
    x[:, 3], x[7, 5], x[9, 6] = 3e38, float("nan"), float("inf")
    mean, invstd, _ = bf.batch_norm_statistics(x, None, None, None, 0.1, 1e-5)
    assert abs(mean[3].item() / 3e38 - 1) < 1e-6 and invstd[3].item() > 0
    assert invstd[5].isnan() and mean[5].isnan() and invstd[6].isnan() and not torch.isfinite(mean[6])
    assert torch.equal(mean[:3], x[0, :3])


@pytest.mark.parametrize("N,K", [(9001, 36), (4099, 7)])
def test_equal_calls_give_equal_bits(backend, N, K):
    g = torch.Generator().manual_seed(N)
    x, dy = (torch.randn(N, K, generator=g) + 3).to(backend), torch.randn(N, K, generator=g).to(backend)
    first = bf.batch_norm_statistics(x, None, None, None, 0.1, 1e-5)
    packed, scale, mn = extq.minmax_pack(x, 2)
    back = bf.batch_norm_backward_packed(dy, None, 0.0, (packed, 2, scale, mn), None, first[0], first[1], [True] * 3)
    for _ in range(3):
        again = bf.batch_norm_statistics(x, None, None, None, 0.1, 1e-5)
        assert all(torch.equal(a, b) for a, b in zip(again, first))
        if back is not None:
            more = bf.batch_norm_backward_packed(dy, None, 0.0, (packed, 2, scale, mn), None, first[0], first[1], [True] * 3)
            assert all(torch.equal(a, b) for a, b in zip(more, back))


def test_malformed_column_vectors_are_refused(backend, monkeypatch):
    """A bias or weight of another length, type or device: the layer leaves it to the framework's routine, and the
    kernels' own entry refuses it; none reads past it."""
    x = torch.randn(9000, 12).to(backend).requires_grad_()
    rm, rv, w = (t.to(backend) for t in (torch.zeros(12), torch.ones(12), torch.ones(12)))

    def framework(*args):
        raise RuntimeError("left to the framework")
    monkeypatch.setattr(bf, "native_batch_norm", framework)
    for bad in (torch.zeros(11).to(backend), torch.zeros(1).to(backend), torch.zeros(13).to(backend), torch.zeros(12).half().to(backend)):
        with pytest.raises(RuntimeError, match="left to the framework"):
            ops.qbatch_norm.apply(x, rm, rv, w, bad, True, 0.1, 1e-5, None)
        with pytest.raises(RuntimeError, match="left to the framework"):
            ops.qbatch_norm.apply(x, rm, rv, bad, w, True, 0.1, 1e-5, None)
    mean, _, mult = bf.batch_norm_statistics(x.detach(), w, None, None, 0.1, 1e-5)
    for bad in (torch.zeros(11).to(backend), torch.zeros(12, dtype=torch.double).to(backend), torch.zeros(24).to(backend)[::2]):
        with pytest.raises(RuntimeError):
            bf.batch_norm_apply(x.detach(), mean, mult, bad)
        assert bf.batch_norm_statistics(x.detach(), w, None, None, 0.1, 1e-5, bad) is None
    if backend.type == "cuda":
        with pytest.raises(RuntimeError):
            bf.batch_norm_apply(x.detach(), mean, mult, torch.zeros(12))
    with pytest.raises(RuntimeError):
        bf.batch_norm_apply(x.detach()[:, :6], mean[:6], mult[:6], None)


@pytest.mark.parametrize("which", ["weight", "bias", "running"])
def test_vectors_of_another_length_are_refused(backend, which):
    """3-D input whose second dimension is not the layer's, or vectors replaced: an error as from torch.nn.BatchNorm1d,
    whose check the native routine leaves out (it would read, and for running statistics write, past their end)."""
    x = torch.randn(6, 40, 16).to(backend)
    layer = layers.QBatchNorm1d(16, affine=which != "running", track_running_stats=which == "running").to(backend).train()
    with pytest.raises(RuntimeError, match="should contain 40 elements not 16"):
        layer(x)
    good = layers.QBatchNorm1d(40).to(backend).train()
    y = good(x)
    assert torch.allclose(y, torch.nn.BatchNorm1d(40).to(backend)(x), atol=1e-5)
    vectors = dict(weight=None, bias=None, running_mean=None, running_var=None)
    for name in (("running_mean", "running_var") if which == "running" else (which,)):
        short = dict(vectors, **{name: torch.ones(39).to(backend)})
        with pytest.raises(RuntimeError, match=name + " should contain 40 elements not 39"):
            bf.native_batch_norm(x, short["weight"], short["bias"], short["running_mean"], short["running_var"], True, 0.1, 1e-5)


@pytest.mark.parametrize("p", [0.0, 0.5, 0.75, 0.3])                   # 1 - p: three powers of two and another number
@pytest.mark.parametrize("bits", [1, 2, 8])
def test_masked_backward_at_the_ends_of_the_range(backend, p, bits):
    """Behind a mask with a subnormal and a huge gradient and rows whose scale has no reciprocal within range (constant ones,
    spreads of 1e-30 and 1e25): the gradients that the separate routines give, to the rounding of the two sums."""
    N, K = 1030, 36
    g = torch.Generator().manual_seed(bits)
    x = torch.randn(N, K, generator=g)
    x[3], x[4], x[5] = 2.0, 1e-30 * x[4], 1e25 * x[5]
    x, dy = x.to(backend), torch.randn(N, K, generator=g).to(backend)
    dy[7, 3], dy[8, 5] = 1e-40, 1e30
    mask = extq.relu_dropout_fwd(torch.ones(N, K).to(backend), p)[1]
    packed, scale, mn = extq.minmax_pack(x, bits)
    mean, invstd = torch.zeros(K).to(backend), torch.ones(K).to(backend)
    got = bf.batch_norm_backward_packed(dy, mask, p, (packed, bits, scale, mn), None, mean, invstd, [True, True, True])
    masked, x_hat = extq.dropout_bwd(dy, mask, p).double(), extq.unpack_bf16param(packed, bits, scale, mn, N, K).double()
    s0, s1 = masked.sum(0), (masked * x_hat).sum(0)
    terms = masked.abs() + masked.abs().sum(0) / N + x_hat.abs() * (masked * x_hat).abs().sum(0) / N
    within = terms < 1e37                                                # the row of 1e25 times its own sum leaves fp32
    assert ((got[0].double() - (masked - s0 / N - x_hat * s1 / N)).abs() <= 1e-5 * terms + 1e-30)[within].all()
    assert within.all(1).sum() >= N - 1
    assert ((got[2].double() - s0).abs() <= 1e-5 * masked.abs().sum(0)).all()


# 512 rows a workgroup: few workgroups, all but one of the 128 groups, one each, one more, and five in one group
@pytest.mark.parametrize("wgs", [17, 127, 128, 129, 513])
def test_the_workgroups_of_a_column_whatever_their_number(backend, wgs):
    """Statistics and the sums of the backward where the last workgroup holds one row and the others unequal values."""
    N, K = (wgs - 1) * 512 + 1, 8
    _check_statistics(backend, "sorted", N, K)
    g = torch.Generator().manual_seed(wgs)
    dy, x = torch.randn(N, K, generator=g).to(backend), torch.randn(N, K, generator=g).to(backend)
    packed, scale, mn = extq.minmax_pack(x, 2)
    mean, invstd = torch.zeros(K).to(backend), torch.ones(K).to(backend)
    sums = bf.batch_norm_backward_packed(dy, None, 0.0, (packed, 2, scale, mn), None, mean, invstd, [False, True, True])
    x_hat = extq.unpack_bf16param(packed, 2, scale, mn, N, K).double()
    for got, terms in ((sums[1], dy.double() * x_hat), (sums[2], dy.double())):
        assert ((got.double() - terms.sum(0)).abs() <= 1e-6 * terms.abs().sum(0)).all()


def _in_groups_of_32(parts, start, add):
    """The order of the kernels that end a reduction: group g takes the workgroups g, g + 32, .. one after the other, then
    the groups follow each other."""
    def chain(items):
        total = start
        for one in items:
            total = add(total, one)
        return total
    groups = [chain(parts[g::32]) for g in range(min(32, len(parts)))]
    total = groups[0]
    for one in groups[1:]:
        total = add(total, one)
    return total


def _rows_per_workgroup(N, K, vec, workgroups, multiple):
    block = 256 * vec
    cols = min(K, block)
    rows = max(-(-N * -(-K // block) // workgroups), -(-4096 // cols))
    turn = 256 // (cols // vec) * multiple
    return -(-rows // turn) * turn


# workgroups fewer than the groups, a few to a group, more than the 16 and 32 that are loaded at once
@pytest.mark.parametrize("N,K", [(1100, 4), (2049, 256), (9000, 256), (2500, 257), pytest.param(50001, 101, marks=pytest.mark.gpu),
                                 pytest.param(169343, 256, marks=pytest.mark.gpu)])
def test_the_sums_of_workgroups_keep_their_order(backend, N, K):
    """Bit for bit: behind a quantiser, statistics that differ in a last bit are other codes."""
    if backend.type == "cpu" and N > 9000:
        pytest.skip("slow on the emulator")
    g = torch.Generator().manual_seed(N)
    x, dy = (torch.randn(N, K, generator=g).to(backend) for _ in range(2))
    L, ptr = _lib.lib(), _checks.ptr
    work = torch.full((bf._scratch_size("exact_bn_work_floats", N, K),), float("nan"), device=backend)
    mean, invstd, mult = torch.empty((3, K), device=backend)
    _lib.check(L.exact_bn_statistics_f32(ptr(x), N, K, 1e-5, 0.1, None, None, None, ptr(work), ptr(mean), ptr(invstd), ptr(mult),
                                         _checks.stream_ptr(x)), "statistics")
    rows = _rows_per_workgroup(N, K, 4, 512, 1) if K % 4 == 0 else _rows_per_workgroup(N, K, 1, 1024, 1)
    workgroups = -(-N // rows)
    parts = work[:workgroups * 3 * K].view(workgroups, 3, K).cpu().numpy()
    assert not np.isnan(parts).any()
    f32 = np.float32

    def join(a, b):
        (na, ma, da), (nb, mb, db) = a, b
        if na == 0:
            return b
        share, d = f32(nb / f32(na + nb)), mb - ma
        df = d.astype(f32)
        return f32(na + nb), ma + d * np.float64(share), da + db + df * df * f32(na * share)
    sets = [(f32(min(rows, N - w * rows)), p[0].astype(np.float64) + p[1].astype(np.float64), p[2]) for w, p in enumerate(parts)]
    _, m, dev = _in_groups_of_32(sets, (f32(0), None, None), join)
    assert np.array_equal(mean.cpu().numpy(), m.astype(f32))
    assert np.array_equal(invstd.cpu().numpy(), f32(1) / np.sqrt(dev / f32(N) + f32(1e-5)))
    if K % 4:
        return
    packed, scale, mn = extq.minmax_pack(x, 2)
    work.fill_(float("nan"))
    sums = torch.empty((2, K), device=backend)
    _lib.check(L.exact_bn_backward_ordered_f32(ptr(dy), None, 0.0, ptr(packed), 2, ptr(scale), ptr(mn), ptr(mean), ptr(invstd), None, N, K,
                                               ptr(work), ptr(sums), None, None, _checks.stream_ptr(x)), "backward")
    workgroups = -(-N // _rows_per_workgroup(N, K, 4, 1024, 4))
    parts = work[:workgroups * 2 * K].view(workgroups, 2, K).cpu().numpy()
    assert not np.isnan(parts).any()
    assert np.array_equal(sums.cpu().numpy(), _in_groups_of_32(list(parts), np.zeros((2, K), f32), lambda a, b: a + b))
