"""Workloads of the package: what its users run, through its public entry points.

A case is a dict of plain values. Its "kind" is one of
  eval        y = layer(x) under torch.no_grad()
  train       y = layer(x); y.backward(g): output and the gradients of x, the
              thresholds and the LUT
  classifier  one training step of the pairwise classifier: logits, cross
              entropy, backward, Adam
  adam        one FusedAdam step over a large layer's parameters

Layer cases carry the input's shape [batch, steps, i] (steps = 0: [batch, i]),
the layer (o, t tables, c comparisons, lut element type), the input's dtype
"x", the route debug mode "debug" ("full" is the module's default: int64
indices and f32 margins kept by every call; "off"; "lazy": uint8 codes), and
for training the STE ("min" or "full"), the surrogate, and "graph": whether
the program replays its step from a HIP graph, as a loop of short steps does.

Inputs and parameters come from the seed alone. x ~ N(0, 1) (image-like, about
80 % zeros, for the classifier), LUT ~ 0.02 N(0, 1) as the module's init
draws it, thresholds near zero as training leaves them.
"""
import math

import torch

from tropnn_amd import FusedAdam, PairwiseLinear, cross_entropy, unit_gradient
from tropnn_amd.examples.emnist import EmnistPairwiseClassifier

DEVICE = "cuda"
DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
DEBUG = {"full": True, "off": False, "lazy": "lazy"}
CLASSES = 10
LR, BETAS, EPS = 1e-3, (0.9, 0.999), 1e-8


def _layer_case(kind, batch, i, o, t, c, *, steps=0, lut="f32", x="f32", debug="off", ste="min",
                surrogate="fast_sigmoid_odd", graph=False):
    case = {"kind": kind, "batch": batch, "steps": steps, "i": i, "o": o, "t": t, "c": c, "lut": lut, "x": x, "debug": debug}
    if kind == "train":
        case.update(ste=ste, surrogate=surrogate, graph=graph)
    return case


def listed():
    named = {
        # serving a small batch, the smallest call: latency, one launch
        "eval_small_b8": _layer_case("eval", 8, 256, 512, 16, 6),
        # bulk inference over f16 reads of the 128-wide layer
        "eval_f16_b8192": _layer_case("eval", 8192, 128, 128, 136, 6, lut="f16"),
        # inference of sequences in bf16, ragged sizes, the module's default debug cache
        "eval_seq_bf16_odd": _layer_case("eval", 7, 300, 250, 100, 5, steps=293, x="bf16", debug="full"),
        # inference through a large layer (1 GiB of f16 LUT)
        "eval_large_f16": _layer_case("eval", 4096, 1024, 4096, 512, 8, lut="f16"),
        # the headline training step: short, replayed from a graph
        "train_c2_graph": _layer_case("train", 512, 128, 128, 136, 6, graph=True),
        # the same layer trained at a large batch, as a GPU this size is used
        "train_b8192": _layer_case("train", 8192, 128, 128, 136, 6),
        # a hidden layer of ordinary width
        "train_wide": _layer_case("train", 4096, 512, 512, 128, 6),
        # sequences with ragged sizes and the module's default debug cache
        "train_seq_odd": _layer_case("train", 12, 300, 250, 100, 5, steps=125, debug="full"),
        # every comparison's gradient, the other surrogate
        "train_full_ste": _layer_case("train", 2048, 128, 128, 136, 6, ste="full", surrogate="izhikevich"),
        # a large layer: f16 reads of a 1 GiB LUT, a 2 GiB f32 LUT gradient
        "train_large_f16": _layer_case("train", 8192, 1024, 4096, 512, 8, lut="f16"),
        # a whole training step of the three-layer classifier
        "classifier_step": {"kind": "classifier", "batch": 512, "i": 784, "hidden": 128, "t": 136, "c": 6},
        # the optimizer's step over a large layer's parameters
        "adam_large": {"kind": "adam", "o": 1024, "t": 256, "c": 8},
    }
    return [dict(case, name=name) for name, case in named.items()]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _width(rng, lo, hi):
    """A feature count: mostly multiples of 16, the rest anything."""
    v = _log_int(rng, lo, hi)
    return max(16, v // 16 * 16) if rng.random() < 0.6 else v


def draw(rng):
    kind = rng.choices(("eval", "train", "classifier", "adam"), (5, 7, 1, 1))[0]
    if kind == "adam":
        return {"kind": "adam", "o": _width(rng, 8, 1024), "t": _log_int(rng, 8, 256), "c": rng.randint(4, 8)}
    if kind == "classifier":
        return {"kind": "classifier", "batch": _log_int(rng, 64, 4096), "i": _width(rng, 64, 1024),
                "hidden": rng.randrange(32, 257, 8), "t": _log_int(rng, 16, 256), "c": rng.randint(4, 7)}
    full = kind == "train" and rng.random() < 0.2
    # work and LUT stay below the largest listed cases'
    most = 1 << (32 if kind == "eval" else 28 if full else 31)
    while True:
        items, i, o = _log_int(rng, 1 if kind == "eval" else 16, 65536), _width(rng, 16, 2048), _width(rng, 8, 4096)
        t, c = _log_int(rng, 8, 512), rng.randint(3, 8)
        if items * t * o <= most and (t << c) * o <= 1 << 26:
            break
    steps = rng.choice((0, 0, 1, rng.randint(2, 64)))
    if steps:
        items = max(1, items // steps)
    return _layer_case(kind, items, i, o, t, c, steps=steps, lut=rng.choice(("f32", "f32", "f16")),
                       x=rng.choice(("f32", "f32", "f32", "bf16", "f16")), debug=rng.choice(("off", "full", "lazy")),
                       ste="full" if full else "min",
                       surrogate=rng.choice(("fast_sigmoid_odd", "fast_sigmoid_odd", "izhikevich")),
                       graph=items * max(1, steps) * t * o <= 1 << 24 and rng.random() < 0.5)


# ---------------------------------------------------------------- inputs


def _generator(seed):
    return torch.Generator(DEVICE).manual_seed(int(seed))


def _parameters(gen, i, o, t, c):
    """Anchors (two different features each), thresholds, LUT."""
    first = torch.randint(0, i, (t, c), generator=gen, device=DEVICE)
    step = torch.randint(1, i, (t, c), generator=gen, device=DEVICE)
    anchors = torch.stack((first, (first + step) % i), dim=-1)
    thresholds = 0.05 * torch.randn(t, c, generator=gen, device=DEVICE)
    lut = torch.randn(t, 1 << c, o, generator=gen, device=DEVICE).mul_(0.02)
    return anchors, thresholds, lut


def _layer_inputs(case, seed):
    gen = _generator(seed)
    shape = (case["batch"], case["steps"], case["i"]) if case["steps"] else (case["batch"], case["i"])
    dtype = DTYPES[case["x"]]
    x = torch.randn(shape, generator=gen, device=DEVICE).to(dtype)
    g = None
    if case["kind"] == "train":
        g = torch.randn(case["batch"], max(1, case["steps"]), case["o"], generator=gen, device=DEVICE).to(dtype)
    return x, g, _parameters(gen, case["i"], case["o"], case["t"], case["c"])


def _fill(layer, anchors, thresholds, lut):
    with torch.no_grad():
        layer.anchors.copy_(anchors)
        layer.thresholds.copy_(thresholds)
        layer.lut.copy_(lut)
    return layer


def _capture(step):
    """`step` after three eager runs on a side stream, as a HIP graph."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(3):
            step()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = step()
    return graph, out


def prepare(case, seed):
    kind = case["kind"]
    if kind == "adam":
        gen = _generator(seed)
        shapes = ((case["t"], case["c"]), (case["t"], 1 << case["c"], case["o"]))
        params = [torch.nn.Parameter(torch.randn(s, generator=gen, device=DEVICE).mul_(0.02)) for s in shapes]
        for p in params:
            p.grad = torch.randn(p.shape, generator=gen, device=DEVICE).mul_(1e-3)
        optimizer = FusedAdam(params, lr=LR, betas=BETAS, eps=EPS)
        optimizer.step()  # the moments exist
        return {"kind": kind, "params": params, "optimizer": optimizer}
    if kind == "classifier":
        gen = _generator(seed)
        x = torch.rand(case["batch"], case["i"], generator=gen, device=DEVICE)
        x = x * (torch.rand(case["batch"], case["i"], generator=gen, device=DEVICE) >= 0.8)
        y = torch.randint(0, CLASSES, (case["batch"],), generator=gen, device=DEVICE)
        with torch.device(DEVICE):
            model = EmnistPairwiseClassifier(input_dim=case["i"], hidden_dim=case["hidden"], num_classes=CLASSES,
                                             comparisons=case["c"], pairwise_tables=case["t"], seed=0).train()
        for layer in model.layers:
            _fill(layer, *_parameters(gen, layer.in_features, layer.out_features, layer.tables, layer.comparisons))
            layer.cache_route_debug = False
        optimizer = FusedAdam(model.parameters(), lr=LR, betas=BETAS, eps=EPS)

        def step():
            optimizer.zero_grad(set_to_none=True)
            logits = model(x)
            loss = cross_entropy(logits, y)
            loss.backward(unit_gradient(loss))
            optimizer.step()
            return logits.detach(), loss.detach()

        graph, out = _capture(step)
        return {"kind": kind, "graph": graph, "outputs": (*out, *(p.grad for p in model.parameters()),
                                                          *(p.detach() for p in model.parameters())),
                "keep": (model, optimizer, x, y)}
    x, g, params = _layer_inputs(case, seed)
    with torch.device(DEVICE):
        layer = PairwiseLinear(case["i"], case["o"], tables=case["t"], comparisons=case["c"],
                               use_min_margin_ste=case.get("ste") != "full",
                               surrogate=case.get("surrogate", "fast_sigmoid_odd"), device_lut_dtype=case["lut"])
    _fill(layer, *params).train(kind == "train")
    layer.cache_route_debug = DEBUG[case["debug"]]
    state = {"kind": kind, "layer": layer, "x": x, "g": g, "debug": case["debug"]}
    if kind == "train":
        x.requires_grad_(True)
        if case["graph"]:
            state["graph"], state["outputs"] = _capture(lambda: _train(state))
    return state


# ---------------------------------------------------------------- one pass


def _debug_outputs(state):
    layer = state["layer"]
    if state["debug"] == "full":
        return (layer._last_indices, layer._last_margins)
    return (layer._last_codes,) if state["debug"] == "lazy" else ()


def _train(state):
    layer, x = state["layer"], state["x"]
    layer.zero_grad(set_to_none=True)
    x.grad = None
    y = layer(x)
    y.backward(state["g"])
    return (y.detach(), x.grad, layer.thresholds.grad, layer.lut.grad, *_debug_outputs(state))


def run(state):
    kind = state["kind"]
    if "graph" in state:
        state["graph"].replay()
        return state["outputs"]
    if kind == "adam":
        optimizer, params = state["optimizer"], state["params"]
        optimizer.step()
        return tuple(t for p in params for t in (p.detach(), optimizer.state[p]["exp_avg"], optimizer.state[p]["exp_avg_sq"]))
    if kind == "eval":
        with torch.no_grad():
            return (state["layer"](state["x"]), *_debug_outputs(state))
    return _train(state)


# ---------------------------------------------------------------- what a pass cannot do without


def _layer_work(items, i, o, t, c, *, lut=4, x=4, train=False, full=False, debug="off"):
    rows = 1 << c
    b = items * (i + o) * x + t * c * (16 + 4) + t * min(items, rows) * o * lut
    flops = items * t * (o + 2 * c)
    if train:
        b += items * (o + i) * x + t * c * 4 + t * rows * o * 4
        flops += items * t * o * (1 + 3 * (c if full else 1))
    b += items * t * (8 + 4 * c) if debug == "full" else items * t if debug == "lazy" else 0
    return b, flops


def work(case):
    if case["kind"] == "adam":
        n = case["t"] * (case["c"] + (case["o"] << case["c"]))
        return {"bytes": 28 * n, "flops": 12 * n}
    if case["kind"] == "classifier":
        b = flops = 0
        for i, o in ((case["i"], case["hidden"]), (case["hidden"], case["hidden"]), (case["hidden"], CLASSES)):
            lb, lf = _layer_work(case["batch"], i, o, case["t"], case["c"], train=True)
            n = case["t"] * (case["c"] + (o << case["c"]))
            b, flops = b + lb + 28 * n, flops + lf + 12 * n
        return {"bytes": b, "flops": flops}
    b, flops = _layer_work(case["batch"] * max(1, case["steps"]), case["i"], case["o"], case["t"], case["c"],
                           lut=2 if case["lut"] == "f16" else 4, x=4 if case["x"] == "f32" else 2,
                           train=case["kind"] == "train", full=case.get("ste") == "full", debug=case["debug"])
    return {"bytes": b, "flops": flops}


def tolerance(case):
    # four times what two correct implementations differ by; each is 0.3e-7 to
    # 2e-7 from 64 bits where its outputs are f32
    if case["kind"] == "adam":
        return {"rel": 5e-7, "max": 1e-4}
    if case["kind"] == "classifier":
        # a last-place change in one layer's output can move a later layer's
        # comparison across zero: that item's rows, and their gradients, change
        return {"rel": 2e-2, "max": 0.9}
    if case["x"] != "f32":
        # output and input gradient rounded to 16 bits: an f32 sum that moves
        # in its last place now and then rounds to the next value
        return {"rel": 2e-4, "max": 1.6e-2} if case["x"] == "bf16" else {"rel": 1e-4, "max": 2e-3}
    # f32 sums over tables and items, in any order
    return {"rel": 2e-6, "max": 1e-4}


# ---------------------------------------------------------------- the same in 64 bits


def _exact_adam(case, seed):
    gen = _generator(seed)
    shapes = ((case["t"], case["c"]), (case["t"], 1 << case["c"], case["o"]))
    params = [torch.randn(s, generator=gen, device=DEVICE).mul_(0.02).double() for s in shapes]
    grads = [torch.randn(s, generator=gen, device=DEVICE).mul_(1e-3).double() for s in shapes]
    out = []
    for p, g in zip(params, grads):
        m, v = torch.zeros_like(p), torch.zeros_like(p)
        for k in (1, 2):
            m = BETAS[0] * m + (1 - BETAS[0]) * g
            v = BETAS[1] * v + (1 - BETAS[1]) * g * g
            p = p - LR / (1 - BETAS[0] ** k) * m / (v.sqrt() / math.sqrt(1 - BETAS[1] ** k) + EPS)
        out += [p, m, v]
    return tuple(out)


def _surrogate(u, name):
    if name == "izhikevich":
        s = torch.sigmoid(u.abs())
        return torch.where(u > 0, -1.0, 1.0) * 2 * s * (1 - s)
    return -0.5 * u.sign() / (1 + u.abs()).square()


def exact(case, seed):
    if case["kind"] == "adam":
        return _exact_adam(case, seed)
    if case["kind"] == "classifier":
        return None  # a later layer's codes are those of an f32 input: 64 bits gives other ones
    x, g, (anchors, thr, lut) = _layer_inputs(case, seed)
    items, i, o, t, c = case["batch"] * max(1, case["steps"]), case["i"], case["o"], case["t"], case["c"]
    scale, rows = 1 / math.sqrt(t), 1 << c
    shape = (case["batch"], max(1, case["steps"]))
    x = x.float().view(items, i)  # margins are f32 by definition: two rounded subtractions
    bits = 2 ** torch.arange(c, device=DEVICE)
    train, full = case["kind"] == "train", case.get("ste") == "full"
    y = torch.zeros(items, o, dtype=torch.float64, device=DEVICE)
    if train:
        g = g.double().view(items, o) * scale
        gx = torch.zeros(items, i, dtype=torch.float64, device=DEVICE)
        gthr = torch.zeros(t, c, dtype=torch.float64, device=DEVICE)
        glut = torch.empty(t, rows, o, dtype=torch.float64, device=DEVICE)
    indices, margins = [], []
    for k in range(t):
        a, b = anchors[k, :, 0], anchors[k, :, 1]
        m = (x[:, a] - x[:, b]) - thr[k]
        code = ((m > 0) * bits).sum(1)
        table = (lut[k].half() if case["lut"] == "f16" else lut[k]).double()
        cur = table[code]
        y += cur
        if case["debug"] != "off":
            indices.append(code)
            margins.append(m)
        if not train:
            continue
        hot = torch.zeros(items, rows, dtype=torch.float64, device=DEVICE)
        hot.scatter_(1, code.unsqueeze(1), 1.0)
        glut[k] = hot.t() @ g
        pick = torch.zeros(items, dtype=torch.long, device=DEVICE)
        for n in range(1, c):  # the first of the smallest |margin|
            best = m.gather(1, pick.unsqueeze(1)).squeeze(1).abs()
            pick = torch.where(m[:, n].abs() < best, n, pick)
        for n in range(c) if full else (pick,):
            n = torch.full_like(pick, n) if full else n
            u = m.gather(1, n.unsqueeze(1)).squeeze(1).double()
            gu = (g * (table[code ^ (1 << n)] - cur)).sum(1) * _surrogate(u, case["surrogate"])
            gthr[k].index_add_(0, n, -gu)
            gx.scatter_add_(1, a[n].unsqueeze(1), gu.unsqueeze(1))
            gx.scatter_add_(1, b[n].unsqueeze(1), -gu.unsqueeze(1))
    y = (y * scale).view(*shape, o)
    debug = ()
    if case["debug"] == "full":
        debug = (torch.stack(indices, 1).view(*shape, t), torch.stack(margins, 1).view(*shape, t, c))
    elif case["debug"] == "lazy":
        debug = (torch.stack(indices, 1).to(torch.uint8).view(*shape, t),)
    if not train:
        return (y, *debug)
    gx = gx.view(*shape, i) if case["steps"] else gx
    return (y, gx, gthr, glut, *debug)
