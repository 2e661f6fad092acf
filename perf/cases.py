"""What this framework is timed on: the calls its users make, from the smallest
to the largest.

A user of this framework compresses activations by hand (`compress`,
`project`), builds a network from its layers (`mlp`), trains GCN and GraphSAGE
models on whole graphs (`gcn`, `sage`), runs a trained model (`evaluate`) and
writes layers of their own on top of the sparse product (`aggregate`).  Sizes
are those of the repository's benchmark configurations and tests, and generic
ones between and beside them (odd and ragged ones among them).  Graphs are
synthetic power-law graphs, features standard normal, as in the benchmark."""
import math

import torch
import torch.nn.functional as F

import exact_amd as exact
from exact_amd import ops
from exact_amd.conf import QuantizationConfig, config
from exact_amd.models import GCN, SAGE
from exact_amd.spmm import qmatmul

MOST_VALUES = 2449029 * 256          # of one activation
DEVICE = torch.device("cuda:0")


def listed():
    return [
        # One hidden activation of a graph of a few thousand nodes: two launches, the cost of a call.
        dict(name="compress_small", kind="compress", rows=4096, cols=128, bits=2, half=False),
        # The headline: one hidden activation of a 169,343-node graph, INT2, saved and restored.
        dict(name="compress_medium", kind="compress", rows=169343, cols=256, bits=2, half=False),
        # Mixed-precision training keeps fp16 activations; a width that is no multiple of anything.
        dict(name="compress_half_ragged", kind="compress", rows=100003, cols=301, bits=4, half=True),
        # Input features wide enough that the random projection is what makes them small: 602 -> 76 and back.
        dict(name="project_wide", kind="project", rows=232965, cols=602, bits=2, kept_frac=0.125),
        # A block of separate Q-layers (linear, batch norm, ReLU, dropout, linear), forward and backward.
        dict(name="mlp_step", kind="mlp", rows=50000, cols=256, hidden=512, out=256, bits=2, kept_frac=1.0),
        # A training step on a graph of a few thousand nodes (Erdos-Renyi size of the plumbing configuration): launches.
        dict(name="gcn_step_small", kind="gcn", nodes=4096, degree=10, features=128, hidden=128, classes=16, layers=2,
             bits=2, batch_norm=False, index_bytes=8, amp=False),
        # The 3-layer INT2 GCN with batch norm and dropout on 169,343 nodes.
        dict(name="gcn_step_medium", kind="gcn", nodes=169343, degree=13.7, features=128, hidden=256, classes=40, layers=3,
             bits=2, batch_norm=True, index_bytes=4, amp=False),
        # The same network under autocast on a smaller graph: fp16 operands throughout.
        dict(name="gcn_step_amp", kind="gcn", nodes=40000, degree=16, features=128, hidden=256, classes=40, layers=3,
             bits=2, batch_norm=True, index_bytes=4, amp=True),
        # 2-layer GraphSAGE on a dense graph with wide features and a projection to an eighth.
        dict(name="sage_step_dense", kind="sage", nodes=232965, degree=113.7, features=602, hidden=256, classes=41, layers=2,
             bits=2, kept_frac=0.125, index_bytes=4),
        # 3-layer GraphSAGE at the largest scale: 2.4 M nodes, 124 M entries, INT1, projection to a quarter.
        dict(name="sage_step_large", kind="sage", nodes=2449029, degree=53.7, features=100, hidden=256, classes=47, layers=3,
             bits=1, kept_frac=0.25, index_bytes=4),
        # A trained model's logits for every node: no compression, only the forward products.
        dict(name="sage_evaluate", kind="evaluate", nodes=100000, degree=50, features=300, hidden=128, classes=47, layers=3,
             index_bytes=4),
        # A layer with learned edge weights: aggregation with gradients for the operand and for every edge value.
        dict(name="learned_edges", kind="aggregate", nodes=60000, degree=30, cols=128, reduce="sum", bits=2, index_bytes=8),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same ranges."""
    kind = rng.choice(["compress", "compress", "project", "mlp", "gcn", "gcn", "sage", "sage", "evaluate", "aggregate"])
    bits = rng.choice([1, 2, 2, 4, 8])
    index_bytes = rng.choice([4, 4, 8])
    if kind == "compress":
        cols = _log_uniform(rng, 16, 1024)
        rows = min(_log_uniform(rng, 500, 2449029), MOST_VALUES // cols)
        return dict(kind=kind, rows=rows, cols=cols, bits=bits, half=rng.random() < 0.3)
    if kind == "project":
        cols = _log_uniform(rng, 64, 602)
        return dict(kind=kind, rows=_log_uniform(rng, 2000, 1000000), cols=cols, bits=bits,
                    kept_frac=rng.choice([0.1, 0.125, 0.2]))
    if kind == "mlp":
        return dict(kind=kind, rows=_log_uniform(rng, 1000, 300000), cols=_log_uniform(rng, 32, 512),
                    hidden=_log_uniform(rng, 64, 512), out=_log_uniform(rng, 16, 512), bits=bits,
                    kept_frac=rng.choice([1.0, 0.25]))
    if kind == "gcn":
        amp, batch_norm = rng.random() < 0.2, rng.random() < 0.5
        # fp16 parameters are too coarse for 255 levels (a row's largest value may wrap): 8 bits are not used with them;
        # and a bias ahead of a batch norm has a gradient that is nothing but the rounding of the kept copy
        return dict(kind=kind, nodes=_log_uniform(rng, 2000, 300000), degree=round(rng.uniform(3, 30), 1),
                    features=_log_uniform(rng, 32, 600), hidden=rng.choice([64, 100, 128, 200, 256]),
                    classes=rng.randint(2, 60), layers=rng.choice([2, 3, 4]), bits=min(bits, 4) if amp or batch_norm else bits,
                    batch_norm=batch_norm, index_bytes=index_bytes, amp=amp)
    if kind == "sage":
        return dict(kind=kind, nodes=_log_uniform(rng, 5000, 700000), degree=round(rng.uniform(8, 110), 1),
                    features=_log_uniform(rng, 50, 602), hidden=rng.choice([64, 100, 128, 200, 256]),
                    classes=rng.randint(2, 60), layers=rng.choice([2, 3]), bits=bits,
                    kept_frac=rng.choice([0.125, 0.25, 1.0]), index_bytes=index_bytes)
    if kind == "evaluate":
        return dict(kind=kind, nodes=_log_uniform(rng, 3000, 500000), degree=round(rng.uniform(5, 100), 1),
                    features=_log_uniform(rng, 50, 602), hidden=rng.choice([64, 128, 256]), classes=rng.randint(2, 60),
                    layers=rng.choice([2, 3]), index_bytes=index_bytes)
    return dict(kind=kind, nodes=_log_uniform(rng, 3000, 200000), degree=round(rng.uniform(5, 60), 1),
                cols=_log_uniform(rng, 16, 256), reduce=rng.choice(["sum", "sum", "mean", "max"]), bits=bits,
                index_bytes=index_bytes)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _generator(seed):
    return torch.Generator(device=DEVICE).manual_seed(seed)


def _graph(nodes, degree, index_bytes, gen, normalise=False):
    """A symmetric power-law graph with about nodes * degree entries, as a
    trainer holds it: CSR with every cached index vector filled in.  Degrees
    have a Pareto tail of exponent 2.1; targets are uniform."""
    raw = torch.rand(nodes, generator=gen, device=DEVICE).clamp_(min=1e-9).pow(-1.0 / 1.1)
    cap = float(max(64, nodes // 16))
    raw.clamp_(max=cap)
    out_degree = (raw * (nodes * degree / 2 / raw.sum())).round().clamp_(min=1, max=cap).long()
    src = torch.repeat_interleave(torch.arange(nodes, device=DEVICE), out_degree)
    dst = torch.randint(0, nodes, (src.numel(),), generator=gen, device=DEVICE)
    keep = src != dst
    src, dst = src[keep], dst[keep]
    key = torch.cat([src * nodes + dst, dst * nodes + src]).unique()
    row, col = torch.div(key, nodes, rounding_mode="floor"), key % nodes
    rowptr = torch.zeros(nodes + 1, dtype=torch.long, device=DEVICE)
    torch.cumsum(torch.bincount(row, minlength=nodes), 0, out=rowptr[1:])
    adj = exact.SparseTensor(rowptr, col, None, (nodes, nodes))
    adj.storage._row = row
    if normalise:
        adj = exact.gcn_norm(adj, add_self_loops=True)
    adj.fill_cache_()
    return adj.to_int32_() if index_bytes == 4 else adj


def _weighted_graph(nodes, degree, index_bytes, gen):
    """A directed graph of exactly round(nodes * degree) entries with a Pareto
    tail of row lengths and a learnable weight on every entry."""
    entries = int(round(nodes * degree))
    weight = torch.rand(nodes, generator=gen, device=DEVICE).clamp_(min=1e-9).pow(-1.0 / 1.1).clamp_(max=float(max(64, nodes // 16)))
    edge = weight.double().cumsum(0)
    row = torch.searchsorted(edge, torch.rand(entries, generator=gen, device=DEVICE, dtype=torch.double) * edge[-1]).clamp_(max=nodes - 1)
    col = torch.randint(0, nodes, (entries,), generator=gen, device=DEVICE)
    adj = exact.SparseTensor.from_edge_index(row, col, None, (nodes, nodes)).fill_cache_()
    if index_bytes == 4:
        adj.to_int32_()
    return adj.set_value(torch.rand(entries, generator=gen, device=DEVICE).requires_grad_())


def _configure(case):
    """The settings a trainer makes once, everything else at its default."""
    config.__dict__.update(QuantizationConfig().__dict__)
    config.activation_compression_bits = [case.get("bits", 2)]
    config.kept_frac = case.get("kept_frac", 1.0)


def prepare(case, seed):
    _configure(case)
    gen = _generator(seed)
    torch.manual_seed(seed)                      # the weights of a model are drawn from torch's own generators
    s = dict(case, seed=seed)
    kind = case["kind"]
    if kind in ("compress", "project"):
        # an activation after a linear layer: zero-mean rows of different spread
        x = torch.randn(case["rows"], case["cols"], generator=gen, device=DEVICE)
        x *= 0.5 + torch.rand(case["rows"], 1, generator=gen, device=DEVICE)
        s["x"] = x.half() if case.get("half") else x
    elif kind == "mlp":
        s["x"] = torch.randn(case["rows"], case["cols"], generator=gen, device=DEVICE).requires_grad_()
        s["gy"] = torch.randn(case["rows"], case["out"], generator=gen, device=DEVICE) / case["rows"]
        net = exact.QMLP([case["cols"], case["hidden"], case["out"]], "batch", bias=False, dropout=0.5)
        s["model"] = net.to(DEVICE).train()
    elif kind == "aggregate":
        s["adj"] = _weighted_graph(case["nodes"], case["degree"], case["index_bytes"], gen)
        s["x"] = torch.randn(case["nodes"], case["cols"], generator=gen, device=DEVICE).requires_grad_()
        s["gy"] = torch.randn(case["nodes"], case["cols"], generator=gen, device=DEVICE)
    else:
        s["adj"] = _graph(case["nodes"], case["degree"], case["index_bytes"], gen, normalise=kind == "gcn")
        s["x"] = torch.randn(case["nodes"], case["features"], generator=gen, device=DEVICE)
        # labels that follow from the features, so that gradients are a signal and not the noise of random labels
        teacher = torch.randn(case["features"], case["classes"], generator=gen, device=DEVICE)
        s["labels"] = (s["x"] @ teacher).argmax(1, keepdim=True)
        shape = (case["features"], case["hidden"], case["classes"], case["layers"])
        net = GCN(*shape, dropout=0.5, batch_norm=case["batch_norm"]) if kind == "gcn" else SAGE(*shape, dropout=0.5)
        s["model"] = exact.QModule(net).to(DEVICE)
        s["model"].train(kind != "evaluate")
    if "model" in s and kind != "evaluate":
        # fp16 gradients of a mean over all nodes would be subnormal: a fixed loss scale, taken out again in the step
        s["loss_scale"] = 4096.0 if case.get("amp") else 1.0
        s["optimizer"] = torch.optim.SGD(s["model"].parameters(), lr=0.01 / s["loss_scale"])
    return s


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(s):
    # Every pass draws the same rounding and dropout noise, as in a run that is meant to be reproduced.
    torch.cuda.manual_seed(s["seed"])
    return globals()["_run_" + s["kind"]](s)


def _run_compress(s):
    x = s["x"]
    quantized = ops.quantize_activation(x, None)
    restored = ops.dequantize_activation(quantized, x.shape)
    packed, _, scale, mn = quantized
    return packed, scale, mn, restored


def _run_project(s):
    x = s["x"]
    quantized, randmat, shape = ops.project_and_quantize(x, None)
    restored = ops.rp2input(ops.dequantize_activation(quantized, shape), x.shape, randmat)
    packed, _, scale, mn = quantized
    return packed, scale, mn, randmat, restored


def _run_mlp(s):
    model, x = s["model"], s["x"]
    s["optimizer"].zero_grad()
    x.grad = None
    y = model(x)
    y.backward(s["gy"])
    s["optimizer"].step()
    return y.detach(), x.grad, [p.grad for p in model.parameters()]


def _run_gcn(s):
    model, x, adj = s["model"], s["x"], s["adj"]
    s["optimizer"].zero_grad()
    if s.get("amp"):
        with torch.autocast("cuda", dtype=torch.float16):
            logits = model(x, adj)
    else:
        logits = model(x, adj)
    # the mean negative log-likelihood of the labels
    loss = -F.log_softmax(logits.float(), dim=-1).gather(1, s["labels"]).mean()
    (loss * s["loss_scale"]).backward() if s.get("amp") else loss.backward()
    s["optimizer"].step()
    return logits.detach(), loss.detach(), [p.grad for p in model.parameters()]


_run_sage = _run_gcn


def _run_evaluate(s):
    with torch.no_grad():
        return s["model"](s["x"], s["adj"])


def _run_aggregate(s):
    x, value = s["x"], s["adj"].storage.value()
    x.grad = value.grad = None
    y = qmatmul(s["adj"], x, reduce=s["reduce"])
    y.backward(s["gy"])
    return y.detach(), x.grad, value.grad


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def work(case):
    kind = case["kind"]
    if kind in ("compress", "project"):
        n, g = case["rows"], case["cols"]
        k = int(case["kept_frac"] * g + 0.999) if kind == "project" else g
        element = 2 if case.get("half") else 4
        # the activation in, the packed codes and the row parameters out and in again, the restored activation out
        moved = n * g * element * 2 + 2 * (n * k * case["bits"] / 8 + 4 * n)
        return {"bytes": moved + (8 * g * k if kind == "project" else 0), "flops": 4.0 * n * g * k if kind == "project" else 0}
    if kind == "mlp":
        n, a, h, b = case["rows"], case["cols"], case["hidden"], case["out"]
        # x and dy in, y and dx out, the hidden activation out and in once in each direction, the weights in and out
        return {"bytes": 4 * n * (2 * a + 2 * b + 4 * h) + 16 * (a * h + h * b), "flops": 6.0 * n * (a * h + h * b)}
    n, nnz, i = case["nodes"], case["nodes"] * case["degree"], case["index_bytes"]
    graph = i * (n + 1 + nnz)
    if kind == "aggregate":
        k = case["cols"]
        arg = 2 * i * n * k if case["reduce"] == "max" else 0
        # forward: x in, y out; backward: dy in, dx out, x again for the edge gradient; values in twice, their gradient out
        return {"bytes": 2 * graph + 12 * nnz + 20 * n * k + arg, "flops": 6.0 * nnz * k}
    widths = [case["features"]] + [case["hidden"]] * (case["layers"] - 1) + [case["classes"]]
    element = 2 if case.get("amp") else 4
    moved = flops = 0.0
    for index, (cin, cout) in enumerate(zip(widths[:-1], widths[1:])):
        narrow = min(cin, cout)
        products = 1 if kind == "gcn" else 2
        directions = 1 if kind == "evaluate" else 3 if index else 2      # the first layer's input wants no gradient
        flops += directions * products * 2.0 * n * cin * cout
        # every layer's input in and its output out; one sparse product each way (the first layer needs none on the way back)
        sparse = 1 if kind == "evaluate" or (index == 0 and kind == "sage") else 2
        flops += sparse * 2.0 * nnz * narrow
        moved += sparse * (graph + (4 * nnz if kind == "gcn" else 0))
        moved += element * n * (cin + cout) * (1 if kind == "evaluate" else 2)
    return {"bytes": moved, "flops": flops}


def tolerance(case):
    """How far two correct implementations of the same precision are apart:
    about four times what the library's own alternatives (sums in CSR order,
    the fp32 matrix-core instruction, layers as chains of separate nodes)
    differ by.  Behind a quantiser, a value within a rounding of a boundary
    may take the neighbouring code, which is what sets "rel" and "max" there."""
    kind = case["kind"]
    if kind == "compress":
        return "exact"                                             # defined to the bit
    if kind == "project":
        return {"rel": 4e-3, "max": 0.9, "differ": 1e-4}           # measured: 9.2e-4, 0.22 (one level), 2e-6
    if kind == "evaluate":
        return {"rel": 1e-6, "max": 1e-5}                          # measured: 1.5e-7, 2.4e-6
    if kind == "aggregate":
        return {"rel": 4e-6, "max": 6e-4}                          # measured: 1e-6, 1.4e-4
    if kind == "mlp":
        return {"rel": 5e-3, "max": 0.12}                          # measured: 1.1e-3, 0.028
    if kind == "sage":
        return {"rel": 4e-3, "max": 0.09}                          # measured: 9.9e-4, 0.022
    if case["amp"]:
        return {"rel": 2.5e-2, "max": 0.4}                         # measured: 6.3e-3, 0.11
    return {"rel": 2.5e-2 if case["batch_norm"] else 1.2e-2, "max": 0.2}     # measured: 6e-3 and 3.2e-3, 0.048
