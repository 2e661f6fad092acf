"""QMLP runs (batch norm ->) ReLU -> dropout ahead of a linear layer in one pass:
against the same layers called one by one."""
import warnings

import pytest
import torch

import exact_amd as exact
from exact_amd import layers, ops
from exact_amd.conf import config
from exact_amd.qsheme import QScheme
from gpu_util import SeededNoise


def _step(backend, net, x, gy, one_pass, before=None):
    config.fuse_epilogue = one_pass
    noise = SeededNoise(5)
    config.noise_source = noise.noise_source
    net = net().to(backend).train()
    if before is not None:
        before(net)
    x = x.to(backend).requires_grad_()
    y = net(x)
    y.backward(gy.to(backend))
    return [y.detach(), x.grad] + [p.grad for p in net.parameters()] + list(net.buffers())


def _net(widths, norm, **kw):
    torch.manual_seed(11)
    return layers.QMLP(widths, norm, **kw)


# below and from 8192 rows on (where the one pass begins), widths of whole octs and not (30, 36), a block behind a block
@pytest.mark.parametrize("norm", ["batch", None])
@pytest.mark.parametrize("p", [0.0, 0.3, 0.5])
@pytest.mark.parametrize("N,widths", [(2, [8, 8, 4]), (33, [16, 24, 40, 8]), (1100, [12, 64, 10]), (50, [20, 30, 16]),
                                      (8191, [4, 16, 4]), (8192, [4, 16, 24, 4]), (8193, [4, 40, 4]), (8200, [4, 36, 4])])
def test_one_pass_equals_the_layers(backend, N, widths, p, norm):
    """Bit for bit: results, gradients, running statistics.  (The sums of a bias gradient meet through atomics from 4096 rows on.)"""
    g = torch.Generator().manual_seed(N)
    x, gy = torch.randn(N, widths[0], generator=g), torch.randn(N, widths[-1], generator=g)
    make = lambda: _net(widths, norm, bias=norm is None and N < 4096, dropout=p)    # noqa: E731
    for one, many in zip(_step(backend, make, x, gy, True), _step(backend, make, x, gy, False)):
        assert torch.isfinite(one).all() and torch.equal(one, many)


def test_what_hooks_and_other_layers_see_stays(backend, monkeypatch):
    calls = []
    real = layers.bn_relu_dropout
    monkeypatch.setattr(layers, "bn_relu_dropout", lambda *a: calls.append(1) or real(*a))
    g = torch.Generator().manual_seed(1)
    x, gy = torch.randn(8192, 4, generator=g), torch.randn(8192, 4, generator=g)
    make = lambda: _net([4, 16, 4], "batch", dropout=0.25)                  # noqa: E731
    _step(backend, make, x[1:], gy[1:], True)                               # too short: the framework's statistics
    config.deterministic_reductions = True                                  # the framework's statistics as well
    _step(backend, make, x, gy, True)
    config.deterministic_reductions = False
    assert calls == []
    _step(backend, make, x, gy, True)
    assert calls == [1]
    seen = []

    def hook(net):
        net[2].register_forward_hook(lambda m, i, o: seen.append(o.shape))

    def backward_hook(net):
        net[3].register_full_backward_hook(lambda m, gi, go: seen.append(go[0].shape))

    def frozen(net):
        net[1].eval()

    class Own(layers.QReLU):
        pass

    def own(net):
        net[2] = Own()
    for change, sights in ((hook, 1), (backward_hook, 2), (frozen, 2), (own, 2)):
        _step(backend, make, x, gy, True, change)
        assert calls == [1] and len(seen) == sights
    config.kept_frac = 0.5                                                  # the next layer projects: no copy to make ahead
    _step(backend, make, x, gy, True)
    assert calls == [1]


@pytest.mark.parametrize("norm", ["batch", None])
def test_training_mode_under_inference_mode(backend, norm):
    """A training-mode block whose results carry no version: nothing is handed over ahead, outputs and running statistics
    are those of the layers one by one.  (8200 rows: sizes that take the one pass elsewhere.)"""
    x = torch.randn(8200, 8, generator=torch.Generator().manual_seed(2)).to(backend)
    got = []
    for one_pass in (True, False):
        config.fuse_epilogue = one_pass
        config.noise_source = SeededNoise(5).noise_source
        net = _net([8, 16, 8], norm, bias=norm is None, dropout=0.5).to(backend).train()
        with torch.inference_mode():
            got.append([net(x), *net.buffers()])
    assert all(torch.equal(one, many) for one, many in zip(*got))


@pytest.mark.parametrize("norm", ["batch", None])
def test_the_consumers_scheme_is_noted(backend, norm):
    """A copy made ahead counts as a quantisation by the layer that takes it, as where that layer makes its own."""
    x = torch.randn(8200, 8, generator=torch.Generator().manual_seed(2)).to(backend)
    for one_pass in (True, False):
        config.fuse_epilogue = one_pass
        net = _net([8, 16, 8], norm, dropout=0.5).to(backend).train()
        QScheme.prev_layer = None
        net(x)
        assert net[-1].scheme is not None and QScheme.prev_layer is net[-1].scheme


@pytest.mark.parametrize("conv", [exact.QGCNConv, exact.QSAGEConv])
def test_the_scheme_of_a_convolution_is_noted(backend, monkeypatch, conv):
    adj = exact.SparseTensor(torch.arange(34).to(backend), torch.arange(33).to(backend), None, (33, 33)).fill_cache_()
    layer = (conv(8, 8, normalize=False) if conv is exact.QGCNConv else conv(8, 8)).to(backend).train()
    scheme = layer.lin_scheme if conv is exact.QGCNConv else layer.scheme
    handed = ops.relu_dropout(torch.randn(33, 8).to(backend), 0.5, for_consumer=True)
    noted = []
    monkeypatch.setattr(QScheme, "note_use", lambda self: noted.append(self))
    layer(handed, adj)
    with_copy = list(noted)
    layer(handed.clone(), adj)
    assert scheme in with_copy and noted == with_copy * 2


@pytest.mark.parametrize("norm", ["batch", None])
def test_a_trace_asks_for_no_sizes(backend, norm):
    """A recorded or compiled block is its layers for every number of rows: nothing in it depends on those it was
    recorded with, and there is no warning that something might."""
    net = _net([8, 16, 8], norm, dropout=0.5).to(backend).eval()
    x = torch.randn(8200, 8).to(backend)
    with warnings.catch_warnings():
        warnings.simplefilter("error", torch.jit.TracerWarning)
        traced = torch.jit.trace(net, x)
    assert torch.equal(traced(x[:7]), net(x[:7]))
    compilations = {}
    for block in (net, torch.nn.Sequential(*net)):                          # as often as the layers one by one
        torch.compiler.reset()
        made = compilations[block] = []
        compiled = torch.compile(block, backend=lambda graph, inputs: made.append(1) or graph.forward, fullgraph=True, dynamic=True)
        for rows in (8200, 7, 8195):
            assert torch.equal(compiled(x[:rows]), net(x[:rows]))
    assert len(compilations[net]) == len(made)
