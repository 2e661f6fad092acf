"""A GraphSAGE layer that is evaluated without gradients does what its
submodules would do: hooks fire, modules put in their place are called,
overridden methods are used, and what the separate operations refuse stays
refused."""
import pytest
import torch

import exact_amd as exact
from exact_amd.conf import config
from exact_amd.layers import QLinear
from exact_amd.sparse import SparseTensor


def _case(backend, cls=exact.QSAGEConv, n=60, cin=24, cout=10):
    config.tall_gemm_min_rows = 1
    g = torch.Generator().manual_seed(n + cin)
    src, dst = torch.randint(0, n, (4 * n,), generator=g), torch.randint(0, n, (4 * n,), generator=g)
    adj = SparseTensor.from_edge_index(dst.to(backend), src.to(backend), None, (n, n))
    return cls(cin, cout).to(backend).eval(), adj, torch.randn(n, cin, generator=g).to(backend)


def _both(layer, x, adj):
    want = layer(x, adj).detach()                  # gradients enabled: the separate operations
    with torch.no_grad():
        return layer(x, adj), want


@pytest.mark.parametrize("name", ["lin_l", "lin_r", "msg_and_aggr_func"])
@pytest.mark.parametrize("kind", ["forward", "pre"])
def test_hooks_fire(backend, name, kind):
    layer, adj, x = _case(backend)
    seen, module = [], getattr(layer, name)
    if kind == "forward":
        module.register_forward_hook(lambda m, args, out: seen.append(name) or out * 2.0)
    else:
        module.register_forward_pre_hook(lambda m, args: seen.append(name))
    got, want = _both(layer, x, adj)
    assert len(seen) == 2 and (got - want).abs().max() < 1e-4


def test_hooks_on_every_module_fire(backend):
    layer, adj, x = _case(backend)
    seen = []
    handle = torch.nn.modules.module.register_module_forward_hook(lambda m, args, out: seen.append(type(m).__name__))
    try:
        with torch.no_grad():
            layer(x, adj)
    finally:
        handle.remove()
    assert sorted(seen) == ["QLinear", "QLinear", "QMatmul", "QSAGEConv"]


def test_a_weight_that_a_pre_hook_makes(backend):
    layer, adj, x = _case(backend)
    torch.nn.utils.weight_norm(layer.lin_l)        # recomputes .weight from weight_g / weight_v ahead of every call
    with torch.no_grad():
        layer.lin_l.weight_g.mul_(3.0)
    got, want = _both(layer, x, adj)
    assert (got - want).abs().max() < 1e-4


def test_parametrised_weight(backend):
    layer, adj, x = _case(backend)

    class Doubled(torch.nn.Module):
        def forward(self, w):
            return 2.0 * w
    torch.nn.utils.parametrize.register_parametrization(layer.lin_r, "weight", Doubled())
    got, want = _both(layer, x, adj)
    assert (got - want).abs().max() < 1e-4


class _Adapter(torch.nn.Module):
    """A low-rank term beside a frozen linear map whose weight it shows."""

    def __init__(self, base):
        super().__init__()
        self.base, self.weight, self.bias = base, base.weight, base.bias
        self.down = torch.nn.Linear(base.in_features, 3, bias=False)
        self.up = torch.nn.Linear(3, base.out_features, bias=False)

    def forward(self, x, quantized=None, randmat=None):
        return self.base(x) + self.up(self.down(x))


class _Bare(torch.nn.Module):
    def forward(self, x, quantized=None, randmat=None):
        return x[:, :10] * 0.5


@pytest.mark.parametrize("name", ["lin_l", "lin_r"])
def test_modules_in_place_of_the_linear_maps(backend, name):
    for make in (lambda m: _Adapter(m), lambda m: _Bare()):
        layer, adj, x = _case(backend)
        setattr(layer, name, make(getattr(layer, name)).to(backend))
        got, want = _both(layer, x, adj)
        assert (got - want).abs().max() < 1e-4


def test_a_subclass_and_an_instance_that_override_a_method(backend):
    class Twice(exact.QSAGEConv):
        def message_and_aggregate(self, adj_t, x, quantized=None, randmat=None):
            return 2.0 * super().message_and_aggregate(adj_t, x, quantized, randmat)

    class Shifted(QLinear):
        def forward(self, input, quantized=None, randmat=None):  # noqa: A002
            return super().forward(input, quantized, randmat) + 1.0

    layer, adj, x = _case(backend, Twice)
    got, want = _both(layer, x, adj)
    assert (got - want).abs().max() < 1e-4
    layer, adj, x = _case(backend)
    shifted = Shifted(24, 10, bias=False).to(backend).eval()
    shifted.load_state_dict(layer.lin_r.state_dict())
    layer.lin_r = shifted
    got, want = _both(layer, x, adj)
    assert (got - want).abs().max() < 1e-4
    layer, adj, x = _case(backend)
    own = layer.lin_l.forward
    layer.lin_l.forward = lambda t: own(t) * 3.0
    got, want = _both(layer, x, adj)
    assert (got - want).abs().max() < 1e-4
    layer, adj, x = _case(backend)
    layer.lin_r.bias = torch.nn.Parameter(torch.ones(10, device=x.device))
    got, want = _both(layer, x, adj)
    assert (got - want).abs().max() < 1e-4


def test_forward_mode_tangents_are_not_dropped(backend):
    """The sparse product has no forward-mode rule: a dual input is refused, with and without no_grad."""
    import torch.autograd.forward_ad as fwad
    layer, adj, x = _case(backend)
    with fwad.dual_level():
        dual = fwad.make_dual(x, torch.ones_like(x))
        for grad in (True, False):
            with torch.set_grad_enabled(grad), pytest.raises(Exception):
                layer(dual, adj)


def test_a_dispatch_mode_sees_the_products(backend):
    from torch.utils._python_dispatch import TorchDispatchMode

    class Count(TorchDispatchMode):
        products = 0

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            self.products += func.overloadpacket in (torch.ops.aten.mm, torch.ops.aten.addmm)
            return func(*args, **(kwargs or {}))

    layer, adj, x = _case(backend)
    with torch.no_grad(), Count() as count:
        layer(x, adj)
    assert count.products == 2
