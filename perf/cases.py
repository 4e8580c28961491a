"""The work that is timed when this framework's speed is measured.

Each case is one call that a user's program makes through the operator API
(``jakal_net``): the forward alone as a serving loop runs it, or the forward and
the backward of a training step, over same-layer propagation (top-k, causal
window, every pair), routing between two layers (top-k and dense routes, there
and back), and the Progressive-B query-block model.  Sizes are those of the
repository's workloads (bench.py), or odd ones beside them; ``draw`` gives more
of the same ranges.

Inputs are what the operators meet inside a model: value rows as a LayerNorm
leaves them (zero mean, unit variance), states and incoming gradients N(0, 1),
weights of the modules' own initialisation, all from the case's seed.  A case
with ``graph`` replays the training step captured into a HIP graph, which is how
a program runs steps whose kernels are shorter than their launches.
"""

from __future__ import annotations

import math
import sys
from pathlib import Path

import torch
from torch.nn import functional as F

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "jakal-net_amd"))

import jakal_net as J  # noqa: E402
from jakal_net.compress import signed_abs_softmax, signed_entmax15  # noqa: E402
from jakal_net.progressive import ProgressiveBConfig, ProgressiveBStep  # noqa: E402

EDGE_COMPRESS = {"softsign": F.softsign, "signed_abs_softmax": signed_abs_softmax, "signed_entmax15": signed_entmax15}


def propagation(mode, batch, nodes, dim, rank, k=0, heads=1, compress="softsign", dtype="f32", train=True, graph=False):
    """A same-layer propagation: mode topk (k sources a row), window (k earlier sources and the row itself) or dense."""
    return dict(op="propagation", mode=mode, batch=batch, nodes=nodes, dim=dim, rank=rank, k=k, heads=heads,
                compress=compress, dtype=dtype, train=train, graph=graph)


def transition(batch, src, dst, dim, rank, k=0, compress="softmax", dtype="f32", train=True, graph=False):
    """Routing from src to dst nodes and back again: k destinations a source row, or (k = 0) all of them."""
    return dict(op="transition", batch=batch, src=src, dst=dst, dim=dim, rank=rank, k=k, compress=compress,
                dtype=dtype, train=train, graph=graph)


def listed():
    return [
        # the query slots of one decoding round: a causal window over all 64 slots, forward only; the smallest call
        dict(name="query_window_infer", **propagation("window", 16, 64, 512, 64, k=63, train=False)),
        # one training step of a block's expanded slots (256 nodes, top-16): many such calls make up a model's step
        dict(name="slots_topk_train", **propagation("topk", 16, 256, 512, 64, k=16)),
        # a sequence of 1024 tokens with a causal window of 64: the ordinary sequence layer, step captured
        dict(name="window_train", **propagation("window", 8, 1024, 384, 32, k=64, graph=True)),
        # top-16 routing between a sequence and a slot layer, both ways, step captured
        dict(name="routes_train", **transition(8, 1024, 256, 512, 64, k=16, graph=True)),
        # the same layers with every route kept, forward only in bf16: a serving pass
        dict(name="routes_dense_bf16_infer", **transition(8, 1024, 256, 512, 64, dtype="bf16", train=False)),
        # the headline training step: 4096 nodes, top-32, fp32
        dict(name="topk_train", **propagation("topk", 16, 4096, 512, 64, k=32)),
        # the same with bf16 layers
        dict(name="topk_bf16_train", **propagation("topk", 16, 4096, 512, 64, k=32, dtype="bf16")),
        # one graph of 4096 nodes answered alone: forward only at batch 1
        dict(name="topk_infer", **propagation("topk", 1, 4096, 512, 64, k=32, train=False)),
        # every pair of 4096 nodes in fp32, training step: the largest
        dict(name="dense_train", **propagation("dense", 16, 4096, 512, 64)),
        # the same with bf16 layers
        dict(name="dense_bf16_train", **propagation("dense", 16, 4096, 512, 64, dtype="bf16")),
        # odd sizes, two heads, row-normalised edges: nothing is a multiple of a tile
        dict(name="ragged_heads_train", **propagation("topk", 3, 1531, 200, 24, k=13, heads=2,
                                                      compress="signed_abs_softmax")),
        # the whole Progressive-B model under bf16 autocast: prefix encoding and query logits
        dict(name="progressive_logits", op="progressive", batch=16, prefix=512, query=64, dim=512, vocab=16384,
             blocks=4),
    ]


LARGEST = 16 * 4096 * 4096  # pairs of the largest listed case


def _spread(rng, low, high):
    """A whole number between low and high, even over the logarithm."""
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _dim(rng):
    """Value widths from 64 to 512: mostly multiples of 32, some of 4, some odd."""
    d = _spread(rng, 64, 512)
    how = rng.random()
    return d // 32 * 32 if how < 0.6 else d // 4 * 4 if how < 0.85 else d


def _rank(rng):
    r = _spread(rng, 8, 64)
    return r // 8 * 8 if rng.random() < 0.75 else r


def draw(rng):
    kind = rng.choice(["topk", "topk", "topk", "window", "window", "dense", "dense", "routes", "routes", "dense_routes",
                       "model"])
    train = rng.random() < 0.65
    dtype = "bf16" if rng.random() < 0.35 else "f32"
    if kind == "model":
        return dict(op="progressive", batch=_spread(rng, 1, 16), prefix=_spread(rng, 70, 512),
                    query=_spread(rng, 8, 64), dim=rng.choice([256, 384, 512]), vocab=rng.choice([4096, 16384]),
                    blocks=rng.choice([1, 2, 4]))
    dim, rank = _dim(rng), _rank(rng)
    if kind in ("routes", "dense_routes"):
        batch, src, dst = _spread(rng, 1, 16), _spread(rng, 64, 2048), _spread(rng, 64, 1024)
        k = min(_spread(rng, 4, 48), src - 1, dst - 1) if kind == "routes" else 0
        if rng.random() < 0.5:
            src, dst = -(-src // 64) * 64, -(-dst // 64) * 64
        return transition(batch, src, dst, dim, rank, k=k, dtype=dtype, train=train,
                          compress=rng.choice(["softmax", "softmax", "signed_abs_softmax", "signed_entmax15"]),
                          graph=train and rng.random() < 0.4)
    batch, nodes = _spread(rng, 1, 16), _spread(rng, 64, 4096)
    if rng.random() < 0.5:
        nodes = min(4096, -(-nodes // 64) * 64)
    heads = rng.choice([1, 1, 1, 2]) if rank <= 32 else 1
    k = min(_spread(rng, 4, 48), nodes - 1) if kind == "topk" else min(_spread(rng, 8, 128), nodes - 1)
    compress = rng.choice(["softsign", "softsign", "signed_abs_softmax", "signed_entmax15"])
    if kind == "dense":
        k = 0
        while batch > 1 and batch * nodes * nodes > LARGEST // 2:
            batch //= 2
        if compress == "signed_entmax15" or heads > 1:  # several passes over the pairs
            batch = max(1, batch // 2)
    return propagation(kind, batch, nodes, dim, rank, k=k, heads=heads, compress=compress, dtype=dtype, train=train,
                       graph=train and kind != "dense" and batch * nodes <= 16384 and rng.random() < 0.4)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _dtype(case):
    return torch.bfloat16 if case["dtype"] == "bf16" else torch.float32


def _normal(g, *shape, dtype=torch.float32):
    return torch.randn(*shape, generator=g, device="cuda").to(dtype)


def _values(g, batch, nodes, dim, dtype):
    return F.layer_norm(_normal(g, batch, nodes, dim), (dim,)).to(dtype)


def _score_weights(g, heads, rank, in_a, in_b):
    """[heads] of (source projection, target projection, core weight, bias): nn.Linear's initialisation of the two
    projections; the core weight and the bias somewhat off their initial one and zero, as after some training."""
    uniform = lambda n, d: (torch.rand(n, d, generator=g, device="cuda") * 2 - 1) / math.sqrt(d)  # noqa: E731
    return [(uniform(rank, in_a), uniform(rank, in_b), 1 + 0.1 * _normal(g, rank), 0.1 * _normal(g, 1)[0])
            for _ in range(heads)]


def _propagation_inputs(case, seed):
    g, B, N, D = _generator(seed), case["batch"], case["nodes"], case["dim"]
    dt = _dtype(case)
    x = dict(state=_normal(g, B, N, dtype=dt), val=_values(g, B, N, D, dt),
             weights=_score_weights(g, case["heads"], case["rank"], D, D))
    if case["train"]:
        x.update(g_state=_normal(g, B, N, dtype=dt), g_val=_normal(g, B, N, D, dtype=dt))
    return x


def _transition_inputs(case, seed):
    g, B, D = _generator(seed), case["batch"], case["dim"]
    dt, sizes = _dtype(case), (case["src"], case["dst"])
    x = dict(state=[_normal(g, B, n, dtype=dt) for n in sizes], val=[_values(g, B, n, D, dt) for n in sizes],
             weights=[_score_weights(g, 1, case["rank"], D, D)[0] for _ in range(2)])
    if case["train"]:
        x.update(g_state=[_normal(g, B, n, dtype=dt) for n in sizes[::-1]],
                 g_val=[_normal(g, B, n, D, dtype=dt) for n in sizes[::-1]])
    return x


def _load(module, weights):
    """The module on the GPU with these (source, target, core, bias) parameters."""
    module = module.to("cuda")
    with torch.no_grad():
        for p, t in zip((module.source_proj.weight, module.target_proj.weight, module.weight, module.bias), weights):
            p.copy_(t)
    return module


def _captured(step):
    """The replay of one call of step, captured after two calls on another stream, and the call's outputs."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(2):
            step()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = step()
    return graph, out


def prepare(case, seed):
    if case["op"] == "progressive":
        return _prepare_model(case, seed)
    return (_prepare_propagation if case["op"] == "propagation" else _prepare_transition)(case, seed)


def _finish(case, step):
    if case["graph"]:
        graph, out = _captured(step)
        return dict(graph=graph, out=out)
    return dict(step=step)


def _prepare_propagation(case, seed):
    x = _propagation_inputs(case, seed)
    heads = [_load(J.LowRankBilinearPairwise(case["dim"], case["rank"]), w) for w in x["weights"]]
    pair = heads[0] if len(heads) == 1 else J.MultiHeadPairwise(heads, aggregate="max")
    common = dict(edge_compress_fn=EDGE_COMPRESS[case["compress"]], implementation="native")
    if case["mode"] == "dense":
        op = J.Propagation(pair, **common)
    elif case["mode"] == "window":
        op = J.SparsePropagation(pair, sparse_type="window", window=case["k"], **common)
    else:
        op = J.SparsePropagation(pair, sparse_type="topk", topk=case["k"], **common)
    train = case["train"]
    state, val = (x[n].requires_grad_(train) for n in ("state", "val"))
    layer = J.Layer(dim=case["dim"], num_nodes=case["nodes"], state=state, val=val)

    def step():
        if not train:
            with torch.no_grad():
                delta = op.compute_delta(layer)
            return dict(delta_state=delta.delta_state, delta_val=delta.delta_val)
        op.zero_grad(set_to_none=True)
        state.grad = val.grad = None
        delta = op.compute_delta(layer)
        torch.autograd.backward([delta.delta_state, delta.delta_val], [x["g_state"], x["g_val"]])
        return dict(delta_state=delta.delta_state.detach(), delta_val=delta.delta_val.detach(), grad_state=state.grad,
                    grad_val=val.grad, grad_weights=[[p.grad for p in _parameters(h)] for h in heads])

    return _finish(case, step)


def _parameters(module):
    return module.source_proj.weight, module.target_proj.weight, module.weight, module.bias


def _prepare_transition(case, seed):
    x = _transition_inputs(case, seed)
    routes = [_load(J.LowRankBilinearRoute(case["dim"], case["dim"], rank=case["rank"]), w) for w in x["weights"]]
    common = dict(route_compress_name=case["compress"], implementation="native")
    there, back = (J.SparseTransition(r, topk=case["k"], **common) if case["k"] else J.Transition(r, **common)
                   for r in routes)
    train = case["train"]
    leaves = [t.requires_grad_(train) for t in x["state"] + x["val"]]
    a, b = (J.Layer(dim=case["dim"], num_nodes=x["state"][i].shape[1], state=x["state"][i], val=x["val"][i])
            for i in range(2))

    def step():
        if not train:
            with torch.no_grad():
                d1, d2 = there.compute_delta(a, b), back.compute_delta(b, a)
            return dict(delta_state=[d1.delta_state, d2.delta_state], delta_val=[d1.delta_val, d2.delta_val])
        there.zero_grad(set_to_none=True)
        back.zero_grad(set_to_none=True)
        for t in leaves:
            t.grad = None
        d1, d2 = there.compute_delta(a, b), back.compute_delta(b, a)
        torch.autograd.backward([d1.delta_state, d2.delta_state, d1.delta_val, d2.delta_val],
                                x["g_state"] + x["g_val"])
        return dict(delta_state=[d.delta_state.detach() for d in (d1, d2)],
                    delta_val=[d.delta_val.detach() for d in (d1, d2)], grad_state=[t.grad for t in x["state"]],
                    grad_val=[t.grad for t in x["val"]],
                    # the logits' bias reaches no softmax: its gradient is 0 up to rounding
                    grad_weights=[[p.grad for p in _parameters(r)[:4 if _bias_matters(case) else 3]] for r in routes])

    return _finish(case, step)


def _bias_matters(case):
    return case["compress"] != "softmax"


def _prepare_model(case, seed):
    cfg = ProgressiveBConfig(vocab=case["vocab"], dim=case["dim"], prefix=case["prefix"], query=case["query"],
                             blocks=case["blocks"])
    with torch.random.fork_rng(devices=[torch.device("cuda")]):
        torch.manual_seed(seed)
        with torch.device("cuda"):
            model = ProgressiveBStep(cfg)
    g = _generator(seed)
    ids = lambda n: torch.randint(0, case["vocab"] - 1, (case["batch"], n), generator=g, device="cuda")  # noqa: E731
    prefix, target = ids(case["prefix"]), ids(case["query"])

    def step():
        with torch.no_grad(), torch.autocast("cuda", dtype=torch.bfloat16):
            return dict(logits=model.query_logits(model.encode_prefix(prefix), target))

    return dict(step=step, model=model, cfg=cfg, prefix=prefix, target=target)


def run(state):
    if "graph" in state:
        state["graph"].replay()
        return state["out"]
    return state["step"]()


# ---------------------------------------------------------------------------
# what a pass cannot do without, and what its results may be off by
# ---------------------------------------------------------------------------
def _edges(case):
    N, k = case["nodes"], case["k"]
    if case["mode"] == "dense":
        return N * N
    if case["mode"] == "topk":
        return N * min(k, N)
    width = min(k + 1, N)
    return N * width - width * (width - 1) // 2


def work(case):
    """Inputs and outputs once; the projections, the scores of the pairs that have to be looked at, the sums over the
    kept pairs, and in training the two gradients of each of these products (of the kept pairs only)."""
    if case["op"] == "progressive":
        B, P, Q, D, V = (case[n] for n in ("batch", "prefix", "query", "dim", "vocab"))
        r, k, exp, cmp = 64, 16, 256, 64
        head = 2 * B * Q * (D * 4 * D + 4 * D * V)
        nodes = case["blocks"] * (P + 5 * exp + 4 * cmp + 3 * P) + 4 * P + 2 * (P + 2 * Q)
        layers = 2 * B * D * (nodes * 2 * r + case["blocks"] * (P * 33 + (P + 3 * exp + 2 * cmp) * k))
        weights = 4 * (2 * V * D + 4 * D * V + 4 * D * D)
        return {"bytes": weights + 2 * B * Q * V, "flops": head + layers}
    size = 2 if case["dtype"] == "bf16" else 4
    B, D, train = case["batch"], case["dim"], case["train"]
    if case["op"] == "propagation":
        N, R = case["nodes"], case["rank"] * case["heads"]
        kept = _edges(case)
        scored = N * N if case["mode"] == "topk" else kept
        rows = B * N * (D + 1) * size
        flops = 2 * B * (N * D * 2 * R + scored * R + kept * D)
        if train:
            flops += 4 * B * (N * D * 2 * R + kept * R + kept * D)
        weights = 2 * R * D * 4
        return {"bytes": rows * (4 if train else 2) + weights * (2 if train else 1), "flops": flops}
    flops = bytes_ = 0
    for s, d in ((case["src"], case["dst"]), (case["dst"], case["src"])):
        kept = s * (min(case["k"], d) if case["k"] else d)
        flops += 2 * B * ((s + d) * D * case["rank"] + s * d * case["rank"] + kept * D)
        if train:
            flops += 4 * B * ((s + d) * D * case["rank"] + kept * case["rank"] + kept * D)
        bytes_ += B * (s + 2 * d) * (D + 1) * size + 2 * case["rank"] * D * 4
        if train:
            bytes_ += B * (2 * d + s) * (D + 1) * size + 2 * case["rank"] * D * 4
    return {"bytes": bytes_, "flops": flops}


def tolerance(case):
    """About four times what the path is off from ``exact`` over the ranges above.  bf16 rows agree to 3e-3 and the
    model's logits too; 32-bit sums to 3e-6.  Where k entries a row are selected, two entries whose scores are equal
    up to rounding may change places, which changes that row by one of its k terms; a signed weight whose score is 0
    up to rounding may change its sign, and the best of several heads, where two are equal, its head."""
    if case["op"] == "progressive":
        return {"rel": 1e-2, "max": 0.05}
    if case["dtype"] == "bf16":
        return {"rel": 2e-2, "max": 0.99}
    if case.get("heads", 1) > 1:
        return {"rel": 1.5e-2, "max": 0.99}
    if case["k"] and case.get("mode") != "window":
        return {"rel": 6e-3, "max": 0.99}
    if case["compress"] == "signed_abs_softmax":
        return {"rel": 1.2e-3, "max": 0.5}
    return {"rel": 1.2e-5, "max": 1e-4}


# ---------------------------------------------------------------------------
# the same results in 64 bits, from plain torch
# ---------------------------------------------------------------------------
def _entmax15(z, keep):
    """1.5-entmax over the kept entries of the last axis: clamp((z - max) / 2 - tau, 0)^2 with tau from the sorted
    prefix sums."""
    z = z.masked_fill(~keep, -math.inf)
    x = (z - z.amax(-1, keepdim=True)) / 2
    with torch.no_grad():
        top = x.sort(-1, descending=True).values
        live = torch.isfinite(top)
        n = torch.arange(1, x.shape[-1] + 1, device=x.device, dtype=x.dtype)
        t = top.masked_fill(~live, 0.0)
        mean, square = t.cumsum(-1) / n, t.square().cumsum(-1) / n
        tau = mean - ((1 - n * (square - mean.square())).clamp_min(0) / n).sqrt()
        size = ((tau <= top) & live).sum(-1, keepdim=True)
        support = x >= top.gather(-1, size - 1)
    n = support.sum(-1, keepdim=True).to(x.dtype)
    xs = x.masked_fill(~support, 0.0)
    mean = xs.sum(-1, keepdim=True) / n
    spread = (((xs - mean) * support).square()).sum(-1, keepdim=True)
    tau = mean - ((1 - spread) / n).clamp_min(0).sqrt()
    return ((x - tau).clamp_min(0) * support).square().masked_fill(~support, 0.0)


def _compressed(scores, keep, kind):
    if kind == "softsign":
        return F.softsign(scores) * keep
    if kind == "softmax":
        return scores.masked_fill(~keep, -math.inf).softmax(-1)
    if kind == "signed_abs_softmax":
        return scores.sign() * scores.abs().masked_fill(~keep, -math.inf).softmax(-1)
    return scores.sign() * _entmax15(scores.abs(), keep)


def _best(scores, k):
    keep = torch.zeros(scores.shape, dtype=torch.bool, device=scores.device)
    return keep.scatter_(-1, scores.topk(min(k, scores.shape[-1]), -1).indices, True)


def _to_bf16(x):
    """x rounded to bf16, with the gradient of x itself."""
    return x + (x.detach().bfloat16().double() - x.detach())


def _scores(rows, keys, weights, unit, bf16):
    """max over the heads of (w * P rows) . (Q keys) + b for weights (Q, P, w, b), and the scores by which rows rank
    their keys.  bf16 layers round the projection weights to bf16, as autocast's nn.Linear does, and rank by the
    products of bf16 operands."""
    out = None
    for Q, P, w, b in weights:
        q = rows @ (_to_bf16(P) if bf16 else P).t() * (w / w.norm().clamp_min(1e-6) if unit else w)
        s = keys @ (_to_bf16(Q) if bf16 else Q).t()
        score = q @ s.transpose(-1, -2) + b
        out = score if out is None else torch.maximum(out, score)
    if bf16:  # one head
        q, s = (t.detach().bfloat16().double() for t in (q, s))
        return out, q @ s.transpose(-1, -2)
    return out, out.detach()


def _exact_propagation(val, state, weights, mode, k, compress, bf16=False):
    n = val.shape[-2]
    s, order = _scores(val, val, weights, True, bf16)
    if mode == "topk":
        keep = _best(order, k)
    else:
        lag = torch.arange(n, device=val.device)[:, None] - torch.arange(n, device=val.device)[None, :]
        keep = (lag >= 0) & (lag <= k) if mode == "window" else torch.ones_like(lag, dtype=torch.bool)
        keep = keep.expand(s.shape)
    e = _compressed(s, keep, compress)
    return (e @ state.unsqueeze(-1)).squeeze(-1), e @ val


def _exact_transition(src_val, src_state, dst_val, weights, k, compress, bf16=False):
    V, U, w, b = weights  # the source side's projection, the target side's, the core weight, the bias
    s, order = _scores(src_val, dst_val, [(U, V, w, b)], False, bf16)
    keep = _best(order, k) if k else torch.ones_like(s, dtype=torch.bool)
    p = (_compressed(s, keep, compress) * F.softplus(src_state).unsqueeze(-1)).transpose(-1, -2)
    return (p @ src_state.unsqueeze(-1)).squeeze(-1), p @ src_val


def _leaf(t):
    return t.detach().double().requires_grad_(True)


def _keeps_bf16(case):
    """Whether bf16 layers are computed as such: those of several heads, and dense ones of other sizes than whole
    8-element rows and 128-wide tiles, are computed in fp32."""
    sizes = [case["dim"]] + ([case["nodes"]] if case["op"] == "propagation" else [case["src"], case["dst"]])
    dense = case["mode"] == "dense" if case["op"] == "propagation" else not case["k"]
    return case.get("heads", 1) == 1 and not (dense and any(n < 128 or n % 8 for n in sizes))


def exact(case, seed):
    if case["op"] == "progressive":
        return _exact_model(case, seed)
    bf16, train = case["dtype"] == "bf16" and _keeps_bf16(case), case["train"]
    if case["op"] == "propagation":
        x = _propagation_inputs(case, seed)
        weights = [[_leaf(p) for p in w] for w in x["weights"]]
        found = {n: [] for n in ("delta_state", "delta_val", "grad_state", "grad_val")}
        for b in range(case["batch"]):
            state, val = _leaf(x["state"][b]), _leaf(x["val"][b])
            ds, dv = _exact_propagation(val, state, weights, case["mode"], case["k"], case["compress"], bf16)
            if train:
                torch.autograd.backward([ds, dv], [x["g_state"][b].double(), x["g_val"][b].double()])
            for n, t in zip(found, (ds.detach(), dv.detach(), state.grad, val.grad)):
                found[n].append(t)
        if not train:
            return {n: torch.stack(found[n]) for n in ("delta_state", "delta_val")}
        grads = [[p.grad for p in w] for w in weights]
        if case["mode"] == "topk" and case["compress"] != "softsign" and case["heads"] == 1:
            grads[0][3] = None  # a row's best scores are of one sign, so that all of them shift alike: 0 up to rounding
        return dict({n: torch.stack(t) for n, t in found.items()}, grad_weights=grads)
    x = _transition_inputs(case, seed)
    weights = [[_leaf(p) for p in w] for w in x["weights"]]
    leaves = {n: [_leaf(t) for t in x[n]] for n in ("state", "val")}
    out = {"delta_state": [], "delta_val": []}
    for i, j in ((0, 1), (1, 0)):
        ds, dv = _exact_transition(leaves["val"][i], leaves["state"][i], leaves["val"][j], weights[i], case["k"],
                                   case["compress"], bf16)
        if train:
            torch.autograd.backward([ds, dv], [x["g_state"][i].double(), x["g_val"][i].double()])
        out["delta_state"].append(ds.detach())
        out["delta_val"].append(dv.detach())
    if train:
        out.update({"grad_" + n: [t.grad for t in v] for n, v in leaves.items()},
                   grad_weights=[[p.grad for p in w[:4 if _bias_matters(case) else 3]] for w in weights])
        if case["k"] and _bias_matters(case):
            for w in out["grad_weights"]:
                w[3] = None  # a row's best logits are of one sign, so that all of them shift alike: 0 up to rounding
    return out


@torch.no_grad()
def _exact_model(case, seed):
    """The Progressive-B forward in 64 bits: parameters by their names in the model."""
    made = _prepare_model(case, seed)
    P, cfg = {n: t.double() for n, t in made["model"].state_dict().items()}, made["cfg"]
    prefix, target = made["prefix"], made["target"]

    def linear(name, x):
        return F.linear(x, P[name + ".weight"], P[name + ".bias"])

    def norm(name, x):
        return F.layer_norm(x, (cfg.dim,), P[name + ".weight"], P[name + ".bias"])

    def score(name):
        return tuple(P[name + end] for end in (".source_proj.weight", ".target_proj.weight", ".weight", ".bias"))

    def stable(name, layer):
        return torch.tanh(layer[0]), norm(name, layer[1])

    def scaled(delta, scale):
        return delta[0] * scale, delta[1] * scale

    def spread(name, layer, mode, k, scale):
        return scaled(_exact_propagation(layer[1], layer[0], [score(name + ".pairwise_fn")], mode, k, "softsign"), scale)

    def route(name, src, dst, scale):
        return scaled(_exact_transition(src[1], src[0], dst[1], score(name + ".route_fn"), cfg.topk, "softmax"), scale)

    def slots(name):
        return tuple(P[name + end].expand(case["batch"], *P[name + end].shape) for end in ("_state", "_val"))

    val = P["embed.weight"][prefix]
    at = torch.linspace(0.0, 1.0, prefix.shape[1], device=val.device).double().unsqueeze(-1)
    val = val + linear("positions.net.2", F.silu(linear("positions.net.0", at)))
    s = stable("s_norm", (linear("state_init", val).squeeze(-1), val))
    for _ in range(cfg.warmup):  # at the default scale of 0 only the stabilisation stays
        s = stable("s_norm", s)
    cmp = None
    for i in range(cfg.blocks):
        n, (alpha, to_b, to_s) = "blocks.%d." % i, cfg.stage(i)
        s = stable(n + "s_norm", spread(n + "s_prop", s, "window", cfg.s_window, cfg.s_scale))
        cmp = stable(n + "cmp_norm", slots(n + "cmp_slot") if cmp is None else cmp)
        exp = route(n + "expand", cmp, slots(n + "exp_slot"), alpha * cfg.b_scale)
        exp = stable(n + "exp_norm", spread(n + "exp_prop", exp, "topk", cfg.topk, alpha * cfg.b_scale))
        s = stable(n + "s_norm", route(n + "b_to_s", exp, s, alpha * to_s * cfg.cross_scale))
        nxt = route(n + "compress", exp, cmp, alpha * cfg.b_scale)
        nxt = route(n + "s_to_b", s, nxt, alpha * to_b * cfg.cross_scale)
        cmp = stable(n + "cmp_norm", spread(n + "cmp_prop", nxt, "topk", cfg.topk, alpha * cfg.b_scale))
    for i in range(cfg.refine):
        s = stable("s_norm", spread("refine.%d" % i, s, "window", cfg.s_window, cfg.refine_scale))
    start = torch.full_like(target[:, :1], case["vocab"] - 1)
    fed = P["embed.weight"][torch.cat([start, target[:, :-1]], dim=1)]
    fed = linear("feedback_proj", norm("feedback_norm", fed))
    q = stable("q_norm", (linear("state_init", fed).squeeze(-1), fed))
    for _ in range(cfg.query_refine):
        q = stable("q_norm", route("q_transition", s, q, cfg.cross_scale))
        q = stable("q_norm", spread("q_prop", q, "window", cfg.query - 1, cfg.s_scale))
    return dict(logits=linear("head.2", F.gelu(linear("head.0", norm("head_norm", q[1])))))
