"""The work that is timed when a kernel or a launch path changes: what a training loop, an inference server and a
pruning run have this framework do, through its public entry points, from calls of a few microseconds up to the
largest layers of the repository's configurations.

Sizes are those of the repository's own configurations, tests and benchmark (batch 64 784 -> 256; batch 256
4096 -> 4096 with hit counts; the ViT-B/16-shaped MLP block; batch 16384 from 4096 inputs; the (128, 2048) x
(2048, 4096) operator call; 4096 x 4096 weights at 10, 3 and 1 % density), odd ones, and, in ``draw``, anything in
between.  Everything is made on the GPU from the seed alone.
"""
import math

import torch

import mamtorch_amd as mt
from mamtorch_amd import sparse
from mamtorch_amd.sparse import prune

DEV = "cuda"

#: products (N * K * M) of the largest call of each kind, which ``draw`` stays below
MOST_TRAIN = 5.9e10
MOST_EVAL = 2.7e11


def listed():
    return [
        # a classifier's first layer on flattened 28 x 28 images, batch 64: the smallest training step
        {"name": "classifier_train", "kind": "layer_train", "n": 64, "k": 784, "m": 256, "splits": 1, "count": False,
         "inputs": "normal", "weights": "kaiming"},
        # a layer of no round size, last batch of an epoch: no dimension is a multiple of anything
        {"name": "ragged_train", "kind": "layer_train", "n": 250, "k": 1001, "m": 517, "splits": 1, "count": False,
         "inputs": "normal", "weights": "kaiming"},
        # the headline layer: training step with hit counts, as a pruning-aware training loop runs it
        {"name": "layer_train_counts", "kind": "layer_train", "n": 256, "k": 4096, "m": 4096, "splits": 1,
         "count": True, "inputs": "normal", "weights": "kaiming"},
        # MLP half of a ViT-B/16 encoder layer on 64 images: training step of the whole block
        {"name": "vit_block_train", "kind": "block_train", "images": 64, "tokens": 197, "hidden": 768,
         "intermediate": 3072, "weights": "kaiming"},
        # the same block serving one image: latency
        {"name": "vit_block_eval_1", "kind": "block_eval", "images": 1, "tokens": 197, "hidden": 768,
         "intermediate": 3072, "weights": "normal"},
        # large-batch inference, values only: the largest call
        {"name": "large_eval", "kind": "layer_eval", "n": 16384, "k": 4096, "m": 4096, "args": False,
         "inputs": "uniform", "weights": "normal"},
        # large-batch inference that keeps argmax / argmin (statistics of the selected weights)
        {"name": "large_eval_args", "kind": "layer_eval", "n": 16384, "k": 4096, "m": 1024, "args": True,
         "inputs": "uniform", "weights": "normal"},
        # the operators under the reference's signature, (in, out) operand: forward and backward
        {"name": "operator_train", "kind": "operator_train", "n": 128, "k": 2048, "m": 4096, "inputs": "normal",
         "weights": "normal"},
        # a layer pruned to 10 %: forward and backward over the CSR weight
        {"name": "sparse_train", "kind": "sparse_train", "n": 256, "k": 4096, "m": 4096, "density": 0.1},
        # a MAM convolution, 3 x 3 windows on 26 x 26 positions: training step
        {"name": "conv_train", "kind": "conv_train", "batch": 32, "channels": 32, "height": 28, "width": 28,
         "filters": 64, "window": 3, "stride": 1},
        # threshold of a layer, then its survivors as CSR: what a pruning run does per layer
        {"name": "prune_layer", "kind": "prune", "m": 4096, "k": 4096, "rate": 0.9, "score": "magnitude"},
        # sum-of-products SpMM over a pruned weight, as the sparse module runs it
        {"name": "spmm", "kind": "spmm", "m": 4096, "k": 4096, "cols": 4096, "density": 0.01, "layout": "csr"},
    ]


def _size(rng, lo, hi):
    """A size between lo and hi, even over the logarithm; half of them round, half as they come."""
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if rng.random() < 0.5:
        step = 64 if v >= 512 else 16 if v >= 64 else 4
        v = max(step, v // step * step)
    return min(max(v, lo), hi)


def draw(rng):
    kind = rng.choice(["layer_train", "layer_train", "layer_train", "layer_eval", "layer_eval", "block_train",
                       "block_eval", "operator_train", "sparse_train", "conv_train", "prune", "spmm"])
    inputs = rng.choice(["normal", "normal", "relu", "uniform"])
    weights = rng.choice(["kaiming", "normal"])
    if kind == "layer_train":
        while True:
            n, k, m = _size(rng, 16, 16384), _size(rng, 256, 4096), _size(rng, 64, 4096)
            if n * k * m <= MOST_TRAIN:
                return {"kind": kind, "n": n, "k": k, "m": m, "splits": rng.choice([1, 1, 1, 4]),
                        "count": rng.random() < 0.5, "inputs": inputs, "weights": weights}
    if kind == "layer_eval":
        while True:
            n, k, m = _size(rng, 1, 16384), _size(rng, 256, 4096), _size(rng, 64, 16384)
            if n * k * m <= MOST_EVAL:
                return {"kind": kind, "n": n, "k": k, "m": m, "args": rng.random() < 0.5, "inputs": inputs,
                        "weights": weights}
    if kind in ("block_train", "block_eval"):
        hidden = rng.choice([192, 384, 768])
        return {"kind": kind, "images": _size(rng, 1, 64), "tokens": rng.choice([50, 65, 197]), "hidden": hidden,
                "intermediate": 4 * hidden, "weights": weights}
    if kind == "operator_train":
        return {"kind": kind, "n": _size(rng, 16, 1024), "k": _size(rng, 256, 4096), "m": _size(rng, 256, 4096),
                "inputs": inputs, "weights": weights}
    if kind == "sparse_train":
        return {"kind": kind, "n": _size(rng, 64, 512), "k": _size(rng, 512, 4096), "m": _size(rng, 512, 4096),
                "density": round(math.exp(rng.uniform(math.log(0.01), math.log(0.15))), 4)}
    if kind == "conv_train":
        side = rng.choice([14, 28, 32])
        return {"kind": kind, "batch": _size(rng, 4, 64), "channels": _size(rng, 8, 64), "height": side,
                "width": side, "filters": _size(rng, 16, 128), "window": rng.choice([3, 3, 5]),
                "stride": rng.choice([1, 1, 2])}
    if kind == "prune":
        return {"kind": kind, "m": _size(rng, 256, 4096), "k": _size(rng, 256, 4096),
                "rate": rng.choice([0.5, 0.7, 0.9, 0.95, 0.99]), "score": rng.choice(["magnitude", "magnitude", "counts"])}
    return {"kind": kind, "m": _size(rng, 256, 4096), "k": _size(rng, 256, 4096), "cols": _size(rng, 64, 4096),
            "density": round(math.exp(rng.uniform(math.log(0.001), math.log(0.3))), 4),
            "layout": rng.choice(["csr", "csr", "coo"])}


# ---- inputs ----------------------------------------------------------------------------------------------------

def _activations(gen, inputs, *shape):
    """normal: what a LayerNorm or a standardised data set hands on; relu: the same behind a ReLU; uniform: U(-1, 1)."""
    if inputs == "uniform":
        return torch.rand(shape, generator=gen, device=DEV) * 2 - 1
    x = torch.randn(shape, generator=gen, device=DEV)
    return x.relu_() if inputs == "relu" else x


def _weights(gen, weights, fan_in, *shape):
    """kaiming: the module's own initial values, U(+-1/sqrt(fan_in)); normal: N(0, 0.02), a trained layer's shape."""
    if weights == "normal":
        return torch.randn(shape, generator=gen, device=DEV) * 0.02
    return (torch.rand(shape, generator=gen, device=DEV) * 2 - 1) / math.sqrt(fan_in)


def _set(layer, gen, weights):
    with torch.no_grad():
        fan_in = layer.weight[0].numel()
        layer.weight.copy_(_weights(gen, weights, fan_in, *layer.weight.shape))
        if layer.bias is not None:
            layer.bias.copy_((torch.rand(layer.bias.shape, generator=gen, device=DEV) * 2 - 1) / math.sqrt(fan_in))
    return layer


def _sparse_weight(gen, m, k, density):
    """A weight of which every row kept the same number of uniformly drawn entries, N(0, 0.02), as torch.sparse_csr."""
    kept = max(1, round(density * k))
    col = torch.rand((m, k), generator=gen, device=DEV).argsort(dim=1)[:, :kept].sort(dim=1)[0]
    values = torch.randn((m * kept,), generator=gen, device=DEV) * 0.02
    crow = torch.arange(m + 1, device=DEV) * kept
    return torch.sparse_csr_tensor(crow, col.reshape(-1), values, size=(m, k))


def prepare(case, seed):
    gen = torch.Generator(device=DEV).manual_seed(int(seed) + 1)
    kind = case["kind"]
    s = {"kind": kind}
    if kind in ("layer_train", "layer_eval"):
        n, k, m = case["n"], case["k"], case["m"]
        train = kind == "layer_train"
        layer = mt.nn.FullyConnected(k, m, bias=True, splits=case.get("splits", 1), device=DEV,
                                     store_args=bool(case.get("count") or case.get("args")) and case.get("splits", 1) == 1,
                                     selection_count_mode="hits")
        s["layer"] = _set(layer, gen, case["weights"]).train(train)
        s["x"] = _activations(gen, case["inputs"], n, k).requires_grad_(train)
        s["args"] = bool(case.get("args"))
        if train:
            s["g"] = torch.randn((n, m), generator=gen, device=DEV)
            s["count"] = bool(case["count"]) and case["splits"] == 1
            if s["count"]:
                layer.reset_selection_count()
    elif kind in ("block_train", "block_eval"):
        block = mt.nn.MAMMlp(case["hidden"], case["intermediate"], device=DEV)
        _set(block.intermediate, gen, case["weights"])
        _set(block.output, gen, case["weights"])
        s["layer"] = block.train(kind == "block_train")
        shape = (case["images"], case["tokens"], case["hidden"])
        s["x"] = _activations(gen, "normal", *shape).requires_grad_(kind == "block_train")
        if kind == "block_train":
            s["g"] = torch.randn(shape, generator=gen, device=DEV)
    elif kind == "operator_train":
        s["a"] = _activations(gen, case["inputs"], case["n"], case["k"]).requires_grad_()
        s["b"] = _weights(gen, case["weights"], case["k"], case["k"], case["m"]).requires_grad_()
        s["g"] = torch.randn((case["n"], case["m"]), generator=gen, device=DEV)
    elif kind == "sparse_train":
        w = _sparse_weight(gen, case["m"], case["k"], case["density"])
        s["crow"], s["col"], s["m"] = w.crow_indices(), w.col_indices(), case["m"]
        s["values"] = w.values().clone().requires_grad_()
        s["a"] = torch.randn((case["n"], case["k"]), generator=gen, device=DEV).requires_grad_()
        s["g"] = torch.randn((case["n"], case["m"]), generator=gen, device=DEV)
    elif kind == "conv_train":
        layer = mt.nn.MAMConv2d(case["channels"], case["filters"], case["window"], stride=case["stride"]).to(DEV)
        s["layer"] = _set(layer, gen, "kaiming").train()
        s["x"] = _activations(gen, "normal", case["batch"], case["channels"], case["height"], case["width"]).requires_grad_()
        out = [(case[side] - case["window"]) // case["stride"] + 1 for side in ("height", "width")]
        s["g"] = torch.randn((case["batch"], case["filters"], *out), generator=gen, device=DEV)
    elif kind == "prune":
        # the quantiles of N(0, 0.02) in a drawn order: how many survive a rate does not depend on the seed
        n = case["m"] * case["k"]
        q = (torch.arange(n, device=DEV, dtype=torch.float64) + 0.5) / n
        w = torch.erfinv(2 * q - 1).mul_(0.02 * math.sqrt(2)).float()
        s["w"] = w[torch.randperm(n, generator=gen, device=DEV)].view(case["m"], case["k"])
        s["rate"] = case["rate"]
        s["score"] = {}
        if case["score"] == "counts":
            # few weights are picked often, most never
            hits = q.pow(8).mul_(1000).int()
            s["score"] = {"counts": hits[torch.randperm(n, generator=gen, device=DEV)].view(case["m"], case["k"])}
    else:
        w = _sparse_weight(gen, case["m"], case["k"], case["density"])
        s["a"] = w if case["layout"] == "csr" else w.to_sparse_coo()
        s["b"] = torch.randn((case["k"], case["cols"]), generator=gen, device=DEV)
    return s


def _train_step(layer, x, g):
    """Forward and backward as a training loop runs them after ``zero_grad(set_to_none=True)``."""
    x.grad = None
    for p in layer.parameters():
        p.grad = None
    y = layer(x)
    y.backward(g)
    return [y.detach(), x.grad] + [p.grad for p in layer.parameters()]


def run(s):
    kind = s["kind"]
    if kind == "layer_train":
        out = _train_step(s["layer"], s["x"], s["g"])
        if s["count"]:
            s["layer"].update_selection_count()
            out += [s["layer"].max_selection_count, s["layer"].min_selection_count]
        return out
    if kind in ("block_train", "conv_train"):
        return _train_step(s["layer"], s["x"], s["g"])
    if kind in ("layer_eval", "block_eval"):
        with torch.no_grad():
            y = s["layer"](s["x"])
        return [y, s["layer"].argmax, s["layer"].argmin] if s.get("args") else y
    if kind == "operator_train":
        s["a"].grad = s["b"].grad = None
        c, argmax, argmin = mt.kernel.v4.fullyconnected(s["a"], s["b"])
        c.backward(s["g"])
        return [c.detach(), argmax, argmin, s["a"].grad, s["b"].grad]
    if kind == "sparse_train":
        s["a"].grad = s["values"].grad = None
        c, argmax, argmin = sparse.SparseFullyConnectedFunction.apply(s["a"], s["values"], s["crow"], s["col"], s["m"])
        c.backward(s["g"])
        return [c.detach(), argmax, argmin, s["a"].grad, s["values"].grad]
    if kind == "prune":
        threshold = prune.layer_threshold(s["w"], s["rate"], **s["score"])
        csr = prune.dense_to_csr(s["w"], threshold, **s["score"])
        return [threshold, csr.crow_indices(), csr.col_indices(), csr.values()]
    return sparse.kernel.v1.cusparsemm(s["a"], s["b"])


# ---- what a pass cannot do without ------------------------------------------------------------------------------

def _layer_work(n, k, m, train, extra_outputs=0):
    """Words read and written once by one layer, and its products: a multiplication and two comparisons each."""
    words = n * k + k * m + m + n * m + extra_outputs * n * m
    if train:
        words += n * m + n * k + k * m + m      # the output gradient; the gradients of input, weight and bias
    return 4 * words, 3 * n * k * m


def work(case):
    kind = case["kind"]
    if kind in ("layer_train", "layer_eval"):
        n, k, m = case["n"], case["k"], case["m"]
        b, f = _layer_work(n, k, m, kind == "layer_train", 2 if case.get("args") else 0)
        if case.get("count") and case["splits"] == 1:
            b += 4 * 2 * 2 * k * m              # both counters read and written
    elif kind in ("block_train", "block_eval"):
        n, h, i = case["images"] * case["tokens"], case["hidden"], case["intermediate"]
        train = kind == "block_train"
        # tokens in, tokens out, both weights; in training the output gradient and the gradients of all of them
        b = 4 * (2 * n * h + 2 * h * i + (2 * n * h + 2 * h * i if train else 0))
        f = 2 * 3 * n * h * i
    elif kind == "operator_train":
        b, f = _layer_work(case["n"], case["k"], case["m"], True, 2)
    elif kind == "sparse_train":
        n, k, m = case["n"], case["k"], case["m"]
        nnz = case["density"] * m * k
        b, f = 12 * nnz + 8 * m + 4 * nnz + 4 * (2 * n * k + 4 * n * m), 3 * n * nnz
    elif kind == "conv_train":
        k = case["window"] ** 2 * case["channels"]
        pos = math.prod((case[side] - case["window"]) // case["stride"] + 1 for side in ("height", "width"))
        image = case["batch"] * case["channels"] * case["height"] * case["width"]
        n, m = case["batch"] * pos, case["filters"]
        b, f = 4 * (2 * image + 2 * n * m + 2 * k * m), 3 * n * k * m
    elif kind == "prune":
        n = case["m"] * case["k"]
        operands = {"magnitude": 1, "counts": 2}[case["score"]]
        b, f = 4 * operands * n + 12 * (1 - case["rate"]) * n, n
    else:
        nnz = case["density"] * case["m"] * case["k"]
        index = 8 if case["layout"] == "csr" else 16
        b = (4 + index) * nnz + 4 * (case["k"] + case["m"]) * case["cols"]
        f = 2 * nnz * case["cols"]
    return {"bytes": b, "flops": f}


def tolerance(case):
    """Outputs and indices of the MAM kernels are exact; gradients and the SpMM are fp32 sums whose order is free.
    Between two runs of one step with its sums in another order: at most 1.7e-7 (2-norm) and 4.9e-6 (one value)."""
    if case["kind"] in ("layer_eval", "prune"):
        return "exact"
    return {"rel": 1e-6, "max": 5e-5}
