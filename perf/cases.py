"""The inference passes whose speed matters, and how much work each of them is.

A pass is what a program that uses this package does once its network is set up: it runs all layers, asks which
rows survived (the challenge's categories) and reads those rows' activations back.  Its answer has a fixed size: a
mark per row, and room for the activations of as many rows as are expected to survive and a quarter more (the first
survivors once more where there are fewer).  Where the features change from pass to pass it hands them over first,
from host memory.  The networks are the three kinds the library meets: layers
with the structure of the challenge's RadiX-Net files, the band layers of the library's own generator, and layers
without structure.

Keys of a case:
  kind      radix: groups of 16 outputs share two 16-wide runs of inputs, strides 16, 32, ... N/2 in turn, every layer
            behind relabellings of its own; radix-common: the same behind one neuron numbering for the whole network, as
            in consecutive layer files; band: the generator's permuted-stride layers; irregular: 1..nnz random inputs
            with random weights per output
  neuron, layers, batch, nnz (entries per row at most)
  survive   share of the rows that are dense enough to live through every layer (features: Bernoulli rows of
            density 0.10 up to what gives that share); irregular layers keep every row alive
  prune     whether rows that died are dropped between the layers
  feed      device: the features lie in the network's buffers already; host: handed over in every pass
"""
import math

import numpy as np
import torch

import graphchallenge21_amd as gc


def _case(name, kind, neuron, layers, batch, nnz=32, survive=0.03, prune=True, feed="device"):
    return {"name": name, "kind": kind, "neuron": neuron, "layers": layers, "batch": batch, "nnz": nnz, "survive": survive,
            "prune": prune, "feed": feed}


def listed():
    return [
        # the smallest useful call: a few layers on a few hundred rows (the package's smoke run)
        _case("small", "band", 1024, 6, 300, survive=0.5),
        # a service that classifies small batches as they come in, from host memory; sizes that fit no tile
        _case("serve-odd", "radix", 1008, 30, 777, survive=0.3, feed="host"),
        # the challenge itself, its 60000 images or a part of them per call, few of which survive, at each of its four
        # widths (its shallowest depth; the widest network cut to a third of it, so that it can be set up often)
        _case("challenge-1024", "radix", 1024, 120, 60000),
        _case("challenge-4096", "radix-common", 4096, 120, 30000),
        _case("challenge-16384", "radix", 16384, 120, 12000),
        _case("challenge-65536", "radix", 65536, 40, 60000),
        # the benchmark's generated networks on live data: cfg0 with its features handed over in the pass, cfg1 with
        # most rows alive to the end, cfg2 and the headline width with every row carried through every layer
        _case("cfg0-host", "band", 1024, 120, 6000, survive=0.67, feed="host"),
        _case("cfg1", "band", 1024, 120, 60000, survive=0.67),
        _case("cfg2-unpruned", "band", 4096, 60, 60000, survive=0.1, prune=False),
        _case("cfg4-unpruned", "band", 65536, 20, 60000, prune=False),
        # layers without structure: the benchmark's width at full batch, and a wider network of odd sizes
        _case("irregular-1024", "irregular", 1024, 64, 60000, nnz=24),
        _case("irregular-odd", "irregular", 3001, 24, 9999, nnz=24, feed="host"),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["radix", "radix", "radix-common", "band", "band", "irregular"])
    if kind == "irregular":
        neuron = _log_uniform(rng, 256, 8192)
    else:
        neuron = _log_uniform(rng, 512, 65536)
        if rng.random() < 0.5:
            neuron = 1 << int(round(math.log2(neuron)))   # the challenge's widths are powers of two
    if kind.startswith("radix"):
        neuron = max(512, neuron // 16 * 16)
    batch = _log_uniform(rng, 64, 60000)
    if rng.random() < 0.25:
        batch = 60000
    most = 60000 * 65536 * 20 // 4                        # of rows x neurons x layers: a quarter of the largest listed case
    layers = min(_log_uniform(rng, 6, 120), max(6, 65536 * 40 // neuron), max(6, most // (batch * neuron)))
    batch = min(batch, most // (layers * neuron))
    nnz = {"band": rng.choice([8, 16, 32, 32]), "irregular": rng.choice([12, 24])}.get(kind, 32)
    prune = rng.random() < 0.75
    survive = rng.choice([0.03, 0.03, 0.3]) if batch * neuron > 1 << 26 else rng.choice([0.03, 0.3, 0.67])
    feed = "host" if batch * neuron <= 1 << 25 and rng.random() < 0.4 else "device"
    c = _case("", kind, neuron, layers, batch, nnz, survive, prune, feed)
    del c["name"]
    return c


def _bias(neuron):
    """The challenge's bias for the width (the next of its widths for sizes in between)."""
    return -0.30 if neuron <= 1024 else -0.35 if neuron <= 4096 else -0.40 if neuron <= 16384 else -0.45


def _densities(case):
    """Densities of the rows: a row lives on if its density exceeds about -bias (the weights of an output add up to 2, so
    a layer doubles the mean, and what is left after the bias has to exceed what went in)."""
    if case["kind"] == "irregular":
        return 0.40, 0.70
    # (by chance also from a little below: narrow networks, and networks that mix their neurons slowly)
    lo, s = 0.10, case["survive"]
    thr = -_bias(case["neuron"]) - (0.018 if case["kind"] == "radix-common" else 4.0 / case["neuron"])
    return lo, min(1.0, (thr - s * lo) / (1.0 - s))


def _radix_layer(rng, n, stride, perm):
    pin, pout = (perm, perm) if perm is not None else (rng.permutation(n).astype(np.int32), rng.permutation(n))
    base = (np.arange(0, n, 16, dtype=np.int32))[:, None]
    run = np.arange(16, dtype=np.int32)[None, :]
    ins = np.sort(pin[np.concatenate([base + run, (base + stride + run) % n], axis=1)], axis=1)
    col = np.empty((n, 32), np.int32)
    col[pout] = np.repeat(ins, 16, axis=0)
    return np.arange(n + 1, dtype=np.int32) * 32, col.reshape(-1), np.full(n * 32, 0.0625, np.float32)


def _irregular_layer(rng, n, kmax):
    """Every output reads 1..kmax distinct inputs; the weights add up to about 2, as 32 of 1/16 do."""
    cand = np.sort(rng.integers(0, n, size=(n, kmax), dtype=np.int32), axis=1)
    keep = np.ones((n, kmax), bool)
    keep[:, 1:] = cand[:, 1:] != cand[:, :-1]
    keep &= rng.random((n, kmax)) < (rng.integers(1, kmax + 1, size=n) / kmax)[:, None]
    keep[:, 0] = True
    rowptr = np.zeros(n + 1, np.int32)
    np.cumsum(keep.sum(axis=1), out=rowptr[1:])
    col = cand[keep]
    val = (rng.uniform(0.5, 1.5, size=len(col)) * (4.0 / kmax)).astype(np.float32)
    return rowptr, col, val


def _answers(case):
    """Rows whose activations a pass reads back."""
    if case["kind"] == "irregular":
        return case["batch"]
    return max(1, min(case["batch"], int(1.25 * case["survive"] * case["batch"])))


def _layers(case, rng):
    """The distinct layers of a network that is set up from arrays, in the order in which they repeat."""
    kind, n, layers = case["kind"], case["neuron"], case["layers"]
    if kind == "irregular":
        return [_irregular_layer(rng, n, case["nnz"]) for _ in range(min(layers, 6))]
    perm = rng.permutation(n).astype(np.int32) if kind == "radix-common" else None
    strides = [16 << k for k in range(int(math.log2(n // 16)))]
    return [_radix_layer(rng, n, s, perm) for s in strides[:layers]]


def prepare(case, seed):
    kind, n, layers, batch = case["kind"], case["neuron"], case["layers"], case["batch"]
    rng = np.random.default_rng(seed)
    net = gc.Network(n, batch, layers, bias=_bias(n))
    if kind == "band":
        net.synth_layers(seed, nnz_per_row=case["nnz"], value=2.0 / case["nnz"])
    else:
        kinds = _layers(case, rng)
        for l in range(layers):
            net.set_layer_csr(l, *kinds[l % len(kinds)])
    net.inspect()
    lo, hi = _densities(case)
    rows = gc.synth_features_host(seed, n, 0, batch, lo, hi) if case["feed"] == "host" else None
    if rows is None:
        net.synth_features(seed, batch, lo, hi)
    else:
        net.set_features_dense(rows)
    return {"net": net, "rows": rows, "prune": case["prune"], "batch": batch, "answers": _answers(case)}


def run(state):
    net = state["net"]
    if state["rows"] is not None:
        net.set_features_dense(state["rows"])
    net.run(prune=state["prune"])
    ids = net.categories()
    survived = np.zeros(state["batch"], bool)
    survived[ids] = True
    return {"survived": survived, "activations": net.activations(np.resize(ids, state["answers"]))}


def exact(case, seed):
    """The layer chain in 64 bits (the inputs are the generators' own, the arithmetic is torch's)."""
    n, layers, batch = case["neuron"], case["layers"], case["batch"]
    if batch * n > 1 << 26:
        return None
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    kinds = [] if case["kind"] == "band" else _layers(case, np.random.default_rng(seed))
    y = torch.from_numpy(gc.synth_features_host(seed, n, 0, batch, *_densities(case))).to(dev, torch.float64).T.contiguous()
    rows = torch.arange(batch, device=dev)
    bias = float(np.float32(_bias(n)))
    for l in range(layers):
        rowptr, col, val = kinds[l % len(kinds)] if kinds else gc.synth_layer_csr(seed, l, n, case["nnz"], 2.0 / case["nnz"])
        length = np.diff(rowptr)
        out = torch.zeros_like(y)
        for k in range(int(length.max())):
            at = np.flatnonzero(length > k)
            i = torch.from_numpy(at).to(dev)
            c = torch.from_numpy(col[rowptr[at] + k].astype(np.int64)).to(dev)
            w = torch.from_numpy(val[rowptr[at] + k].astype(np.float64)).to(dev)
            out[i] += w[:, None] * y[c]
        out += bias
        if (out.amax(dim=0).abs() < 1e-5).any():
            return None   # a row on the edge of dying: rounding decides whether it is among the answers
        y = out.clamp_(0.0, 32.0)
        if case["prune"]:
            live = (y != 0).any(dim=0)
            y, rows = y[:, live].contiguous(), rows[live]
    live = (y != 0).any(dim=0)
    ids = rows[live].cpu().numpy()
    survived = np.zeros(batch, bool)
    survived[ids] = True
    return {"survived": survived, "activations": np.resize(y[:, live].T.cpu().numpy(), (_answers(case), n))}


def work(case):
    """Bytes: the features and the layers' entries (index and weight) in, the marks and the answered rows' activations out.
    Operations: a multiply-add per entry and row that has to be carried - with pruning the first layer's and the
    survivors' - and, in radix layers, per group of outputs that are the same sum, not per output."""
    n, layers, batch = case["neuron"], case["layers"], case["batch"]
    per_row = case["nnz"] / 2.0 if case["kind"] == "irregular" else float(case["nnz"])
    alive = batch * (1.0 if case["kind"] == "irregular" else case["survive"])
    answers = _answers(case)
    distinct_layers = min(layers, 6) if case["kind"] == "irregular" else layers
    rows = batch + (layers - 1) * (alive if case["prune"] else batch)
    sums = n / 16.0 if case["kind"].startswith("radix") else float(n)
    nbytes = 4.0 * n * batch + 8.0 * n * per_row * distinct_layers + 4.0 * n * answers + batch
    return {"bytes": nbytes, "flops": 2.0 * sums * per_row * rows}


def tolerance(case):
    """Every path adds an output's inputs in ascending input index in 32-bit floats, so results are the same bits."""
    return "exact"
