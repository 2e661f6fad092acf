"""A dense product answers from the weights as they are when it runs: writes
that no version counter sees (moving averages and broadcasts through `.data`),
weights that have none (inference tensors), other streams, captured graphs."""
import pytest
import torch

import exact_amd as exact
from exact_amd.conf import config
from exact_amd.cpp_extension import backward_func as bf
from exact_amd.sparse import SparseTensor


def _ring(n, device):
    i = torch.arange(n)
    return SparseTensor.from_edge_index(torch.cat([i, i]).to(device), torch.cat([(i + 1) % n, (i + 5) % n]).to(device), None, (n, n))


def _plain(layer, x, adj):
    """The layer in float64 by dense products."""
    rowptr, col, _ = adj.csr()
    n = x.shape[0]
    dense = torch.zeros(n, n, dtype=torch.double, device=x.device)
    row = torch.repeat_interleave(torch.arange(n, device=x.device), rowptr[1:] - rowptr[:-1])
    dense.index_put_((row, col), torch.ones(col.numel(), dtype=torch.double, device=x.device), accumulate=True)
    dense /= dense.sum(1, keepdim=True)
    xd = x.double()
    return (dense @ xd) @ layer.lin_l.weight.double().t() + layer.lin_l.bias.double() + xd @ layer.lin_r.weight.double().t()


@pytest.mark.parametrize("transposed", [True, False])
def test_product_follows_a_write_through_data(backend, transposed):
    config.tall_gemm_min_rows = 1
    g = torch.Generator().manual_seed(1)
    x = torch.randint(-4, 5, (70, 24), generator=g).float().to(backend)
    w = torch.nn.Parameter(torch.randint(-4, 5, (40, 24) if transposed else (24, 40), generator=g).float().to(backend))
    with torch.no_grad():
        for factor in (1.0, 3.0, -2.0):                     # integers: every product is exact
            w.data.mul_(factor)
            assert torch.equal(bf.tall_matmul(x, w, transposed=transposed), x.mm(w.t() if transposed else w))
    w.data = w.data + 1.0                                   # another storage under the same Parameter
    with torch.no_grad():
        assert torch.equal(bf.tall_matmul(x, w, transposed=transposed), x.mm(w.t() if transposed else w))


@pytest.mark.parametrize("cin,cout", [(32, 12), (12, 32)])
def test_evaluation_follows_a_write_through_data(backend, cin, cout):
    config.tall_gemm_min_rows = 1
    g = torch.Generator().manual_seed(2)
    layer = exact.QSAGEConv(cin, cout).to(backend).eval()
    adj, x = _ring(90, backend), torch.randn(90, cin, generator=g).to(backend)
    for step in range(3):
        with torch.no_grad():
            got = layer(x, adj)
            assert (got.double() - _plain(layer, x, adj)).abs().max() < 1e-4
            for p in layer.parameters():
                p.data.mul_(0.5).add_(0.3)                  # a moving average, as trainers write it


def test_evaluation_with_inference_tensors(backend):
    config.tall_gemm_min_rows = 1
    with torch.inference_mode():
        layer = exact.QSAGEConv(16, 8).to(backend).eval()
        adj, x = _ring(50, backend), torch.randn(50, 16).to(backend)
        assert layer.lin_l.weight.is_inference()
        first = layer(x, adj)
        assert (first.double() - _plain(layer, x, adj)).abs().max() < 1e-4
        layer.lin_l.weight.mul_(2.0)
        assert (layer(x, adj).double() - _plain(layer, x, adj)).abs().max() < 1e-4
    with torch.no_grad():                                   # made under inference mode, used outside it
        assert (layer(x, adj).double() - _plain(layer, x, adj)).abs().max() < 1e-4


@pytest.mark.gpu
def test_evaluation_on_two_streams(cuda):
    """The weights written on one stream, read by evaluations on two others that wait for that write only."""
    config.tall_gemm_min_rows = 1
    layer = exact.QSAGEConv(64, 32).to(cuda).eval()
    adj, x = _ring(3000, cuda), torch.randn(3000, 64, device=cuda)
    streams, results = [torch.cuda.Stream(), torch.cuda.Stream()], []
    with torch.no_grad():
        layer(x, adj)
        for step in range(6):
            for p in layer.parameters():
                p.data.add_(0.25)
            want = _plain(layer, x, adj)
            for s in streams:
                s.wait_stream(torch.cuda.current_stream())
                with torch.cuda.stream(s):
                    results.append((layer(x, adj), want))
            for s in streams:
                torch.cuda.current_stream().wait_stream(s)
    torch.cuda.synchronize()
    for got, want in results:
        assert (got.double() - want).abs().max() < 1e-3


@pytest.mark.gpu
def test_captured_evaluation_reads_the_weights_of_its_replay(cuda):
    config.tall_gemm_min_rows = 1
    layer = exact.QSAGEConv(64, 32).to(cuda).eval()
    adj, x = _ring(3000, cuda), torch.randn(3000, 64, device=cuda)
    adj.fill_cache_()
    with torch.no_grad():
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            layer(x, adj)
        torch.cuda.current_stream().wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = layer(x, adj)
        for step in range(5):
            for p in layer.parameters():
                p.data.mul_(0.9).add_(0.1)
            eager = layer(x, adj)                           # the program's own work between the replays
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, eager)
            assert (out.double() - _plain(layer, x, adj)).abs().max() < 1e-3
