"""The work a user of loopback_amd has it do, as measurable cases through its public entry points.

Three kinds of program stand behind them:
  * the Loopback read in a layer loop (`loopback_amd.chain`: K shared blocks x R iterations, one stacked write and one
    read per block application): evaluation (no gradients), the same replayed from one HIP graph, and training
    (forward, backward, every gradient); in the stacked layout with stored or online scores and in the list layout;
  * one transformer block of the language model around the read (`loopback_amd.lm.Block`), forward and backward;
  * the language model whole (`loopback_amd.lm.LoopbackLM`): prefill to logits, and loss with every gradient.

Sizes are the repository's configurations 1-5 and its tests' (odd widths, ragged token counts, more than 64 block
applications), the query one that has been trained (at its zero initialisation every read is its prior).
"""
from __future__ import annotations

import math

import torch

from loopback_amd import chain, lm
from loopback_amd.chain import ChainConfig

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
BETA, EPS, Q_STD = 0.75, 1e-6, 0.25


def _chain(name, kind, d, K, R, b, t, dtype, mode="scores"):
    return {"name": name, "kind": kind, "d": d, "K": K, "R": R, "b": b, "t": t, "dtype": dtype, "mode": mode}


def _lm(name, kind, b, t, d=768, heads=12, vocab=32000, P=2, K=4, R=4, C=2):
    return {"name": name, "kind": kind, "d": d, "heads": heads, "vocab": vocab, "P": P, "K": K, "R": R, "C": C,
            "b": b, "t": t, "dtype": "bf16"}


def listed() -> list[dict]:
    return [
        # a short prompt served from a captured graph: latency and the number of launches are everything
        _chain("graph_eval_t128", "graph_eval", 768, 2, 4, 1, 128, "bf16"),
        # configuration 1: a small fp32 evaluation called eagerly
        _chain("eval_c1_fp32", "eval", 768, 2, 4, 2, 256, "fp32"),
        # configuration 2: an ordinary bf16 evaluation batch
        _chain("eval_c2", "eval", 768, 2, 4, 8, 2048, "bf16"),
        # an evaluation with more iterations than trained: 72 block applications, the last reads over more than 64
        _chain("eval_extra_iterations", "eval", 768, 4, 18, 2, 2048, "bf16"),
        # configuration 3: an ordinary training pass
        _chain("train_c3", "train", 1024, 3, 4, 8, 2048, "bf16"),
        # configuration 4: the largest training pass, the headline
        _chain("train_c4", "train", 2048, 4, 8, 8, 2048, "bf16"),
        # fp32 training without the score table (the scores formed as the sources stream), a ragged batch
        _chain("train_fp32_online", "train", 1024, 3, 4, 3, 1365, "fp32", "stack"),
        # the list layout (one tensor per update), in fp16 mixed precision
        _chain("train_list_fp16", "train", 1024, 2, 4, 4, 1024, "fp16", "list"),
        # a width the vector row layout does not take (odd), ragged tokens
        _chain("train_odd_width", "train", 1001, 3, 4, 3, 683, "bf16"),
        # one transformer block of configuration 5 (norms, rotary attention, SwiGLU), forward and backward
        _lm("block_c5", "block", 8, 2048),
        # prefill of configuration 5's model: two sequences of 4096 to their logits
        _lm("prefill_c5", "prefill", 2, 4096),
        # configuration 5: loss and every gradient of the model's training step
        _lm("lm_train_c5", "lm_train", 8, 2048),
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def _cost(c: dict) -> float:
    """Rough bytes a case's pass moves, to keep a drawn case below the largest listed one."""
    if c["kind"] in ("graph_eval", "eval", "train"):
        N = c["K"] * c["R"]
        per = N * N / 2 + 4 * N
        if c["kind"] == "train":
            per *= 6 if c["mode"] == "list" else 3
        slow = 8 if c["d"] % 8 or N > 64 else 1
        return per * c["b"] * c["t"] * c["d"] * (4 if c["dtype"] == "fp32" else 2) * slow
    layers = 1 if c["kind"] == "block" else c["P"] + c["K"] * c["R"] + c["C"]
    tok = c["b"] * c["t"]
    per = 120 * c["d"] * layers + (0 if c["kind"] == "block" else 16 * c["vocab"])
    return 2 * tok * per * (1 if c["kind"] == "prefill" else 3)


def draw(rng) -> dict:
    """One more case of the same ranges."""
    limit = max(_cost(c) for c in listed() if c["kind"] == "train")
    while True:
        kind = rng.choice(["graph_eval", "eval", "eval", "train", "train", "train", "block", "prefill", "lm_train"])
        if kind in ("graph_eval", "eval", "train"):
            K, R = rng.randint(1, 4), rng.randint(2, 8)
            if kind == "eval" and rng.random() < 0.25:
                K, R = 4, rng.randint(17, 20)                       # extra iterations
            if kind != "graph_eval" and rng.random() < 0.25:
                d = _log_int(rng, 96, 2048)                         # any width, odd ones among them
            else:
                d = 8 * _log_int(rng, 12, 256)                      # 96 .. 2048
            T = _log_int(rng, 1 if kind == "graph_eval" else 64, 4096 if kind == "graph_eval" else 16384)
            b = rng.randint(1, 8)
            c = {"kind": kind, "d": d, "K": K, "R": R, "b": b, "t": max(1, T // b),
                 "dtype": rng.choice(["bf16", "bf16", "fp16", "fp32"]),
                 "mode": rng.choice(["scores", "scores", "stack", "list"])}
            if K * R > 64 and c["mode"] == "scores" and rng.random() < 0.5:
                c["mode"] = "stack"
        else:
            heads = rng.choice([4, 8, 12, 16])
            c = _lm(None, kind, rng.randint(1, 8), _log_int(rng, 64, 2048), d=64 * heads, heads=heads,
                    vocab=rng.choice([4096, 16384, 32000]), P=rng.randint(0, 2), K=rng.randint(1, 4),
                    R=rng.randint(2, 4), C=rng.randint(0, 2))
            del c["name"]
        if _cost(c) <= limit:
            return c


# ---------------------------------------------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------------------------------------------
def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _chain_inputs(case, seed):
    """h0 and the blocks' updates N(0, 1) in the updates' dtype, the trained queries and the loss weights in fp32."""
    dev = _device()
    gen = torch.Generator(device=dev).manual_seed(seed)
    shape, N, dtype = (case["b"], case["t"], case["d"]), case["K"] * case["R"], DTYPES[case["dtype"]]
    h0 = torch.randn(shape, generator=gen, device=dev).to(dtype)
    D = [torch.randn(shape, generator=gen, device=dev).to(dtype) for _ in range(N)]
    Q = torch.randn((N - 1, case["d"]), generator=gen, device=dev) * Q_STD
    G = torch.randn(shape, generator=gen, device=dev) if case["kind"] == "train" else None
    return h0, D, Q, G


def _block_shapes(prefix, d, inter):
    return {f"{prefix}attn_norm.weight": (d,), f"{prefix}attn.qkv.weight": (3 * d, d), f"{prefix}attn.o.weight": (d, d),
            f"{prefix}mlp_norm.weight": (d,), f"{prefix}mlp.gate_up.weight": (2 * inter, d),
            f"{prefix}mlp.down.weight": (d, inter)}


def _lm_config(case):
    return lm.LMConfig(hidden_size=case["d"], num_heads=case["heads"], vocab_size=case["vocab"], prelude=case["P"],
                       loop_blocks=case["K"], loops=case["R"], coda=case["C"], beta=BETA)


def _intermediate(d):
    return 256 * ((int(d * 4 * 2 / 3) + 255) // 256)


def _weights(case, seed):
    """Weights of a block ('block') or of the whole model: matrices N(0, 0.02^2), norm gains about 1, in bf16."""
    dev, d = _device(), case["d"]
    gen = torch.Generator(device=dev).manual_seed(seed)
    inter = _intermediate(d)
    if case["kind"] == "block":
        shapes = _block_shapes("", d, inter)
    else:
        shapes = {"embed.weight": (case["vocab"], d)}
        for part, count in (("prelude", case["P"]), ("middle", case["K"]), ("coda", case["C"])):
            for i in range(count):
                shapes.update(_block_shapes(f"{part}.{i}.", d, inter))
        shapes.update({"norm.weight": (d,), "head.weight": (case["vocab"], d),
                       "read.query": (case["K"] * case["R"] - 1, d)})
    out = {}
    for name, shape in shapes.items():
        w = torch.randn(shape, generator=gen, device=dev)
        w = 1 + 0.1 * w if name.endswith("norm.weight") else w * (Q_STD if name == "read.query" else 0.02)
        out[name] = w.bfloat16()
    return out


def _lm_inputs(case, seed):
    dev = _device()
    gen = torch.Generator(device=dev).manual_seed(seed + 1)
    shape = (case["b"], case["t"])
    if case["kind"] != "block":
        return torch.randint(0, case["vocab"], shape, generator=gen, device=dev)
    x = torch.randn((*shape, case["d"]), generator=gen, device=dev).bfloat16()
    return x, torch.randn((*shape, case["d"]), generator=gen, device=dev).bfloat16()


# ---------------------------------------------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------------------------------------------
def prepare(case: dict, seed: int) -> dict:
    kind = case["kind"]
    if kind in ("graph_eval", "eval", "train"):
        cfg = ChainConfig("case", case["d"], case["K"], case["R"], case["b"], case["t"], DTYPES[case["dtype"]],
                          kind == "train", beta=BETA, eps=EPS)
        h0, D, Q, G = _chain_inputs(case, seed)
        state = {"kind": kind, "cfg": cfg, "h0": h0, "D": D, "Q": Q, "G": G, "mode": case["mode"]}
        if kind == "graph_eval":
            state["graph"], state["out"] = chain.capture_forward(cfg, h0, D, Q, case["mode"])
        else:
            state["cell"] = chain.make_cell(cfg, Q)
        return state
    cfg, dev = _lm_config(case), _device()
    model = (lm.Block(cfg) if kind == "block" else lm.LoopbackLM(cfg)).to(device=dev, dtype=torch.bfloat16)
    model.load_state_dict(_weights(case, seed))
    state = {"kind": kind, "model": model, "in": _lm_inputs(case, seed)}
    if kind == "block":
        state["in"][0].requires_grad_()
    return state


def _grads(model):
    return {name: p.grad for name, p in model.named_parameters()}


def run(state: dict):
    kind = state["kind"]
    if kind == "graph_eval":
        state["graph"].replay()
        return state["out"]
    if kind in ("eval", "train"):
        h, _, grads = chain.run_chain(state["cfg"], state["h0"], state["D"], state["Q"], state["G"], state["mode"],
                                      cell=state["cell"])
        return h if grads is None else [h, grads["h0"], grads["query"], *grads["D"]]
    model = state["model"]
    if kind == "prefill":
        with torch.no_grad():
            return model.head(model.hidden(state["in"]))
    model.zero_grad(set_to_none=True)
    if kind == "block":
        x, g = state["in"]
        x.grad = None
        y = model(x)
        y.backward(g)
        return {"y": y.detach(), "x": x.grad, **_grads(model)}
    loss = model(state["in"])
    loss.backward()
    return {"loss": loss.detach(), **_grads(model)}


def work(case: dict) -> dict:
    """Every call's inputs read once and its outputs written once: for the layer loop, per block application the
    block's own add (3 rows), the write (h, x in; the update out), the read (its sources and base in; the state out)
    and in training their gradients (a read: its sources and output gradient; an update: its reads' output gradients
    and itself in, its two gradients out; the two gradients of x added). Weights and activations for the model."""
    d, tok = case["d"], case["b"] * case["t"]
    N = case["K"] * case["R"]
    if case["kind"] in ("graph_eval", "eval", "train"):
        S2 = N * (N + 1) // 2 - 1                              # source visits of the reads
        rows = 3 * N + 3 * N + S2 + 2 * (N - 1)
        flops = 2 * d * tok * 2 * S2                           # scores and weighted sums
        if case["kind"] == "train":
            rows += (S2 + N - 1) + (S2 + N + 2 * N) + 3 * N
            flops += 2 * d * tok * 4 * S2
        return {"bytes": rows * tok * d * (4 if case["dtype"] == "fp32" else 2), "flops": flops}
    inter = _intermediate(d)
    layer = 4 * d * d + 3 * d * inter
    layers = 1 if case["kind"] == "block" else case["P"] + N + case["C"]
    flops = layers * (2 * layer * tok + 2 * 2 * case["b"] * case["t"] ** 2 * d / 2)   # causal: half the scores
    rows = layers * 3 * d
    params = layer
    if case["kind"] != "block":
        flops += 2 * tok * d * case["vocab"]
        params = (case["P"] + case["K"] + case["C"]) * layer + 2 * case["vocab"] * d
        S2 = N * (N + 1) // 2 - 1
        rows += d * (3 * N + S2 + 2 * (N - 1))
        if case["kind"] == "prefill":
            rows += case["vocab"]
    if case["kind"] != "prefill":
        flops, rows, params = 3 * flops, 3 * rows, 3 * params
    return {"bytes": 2 * (rows * tok + params), "flops": flops}


def tolerance(case: dict) -> dict:
    """About four times the distance between each path and the exact result at the same inputs."""
    if case["kind"] in ("prefill", "lm_train"):
        return {"rel": 6e-2}
    if case["kind"] == "block":
        return {"rel": 2e-2}
    return {"rel": {"fp32": 6e-6, "fp16": 4e-3, "bf16": 3.5e-2}[case["dtype"]]}


# ---------------------------------------------------------------------------------------------------------------
# the same in 64 bits, in plain torch
# ---------------------------------------------------------------------------------------------------------------
def _read64(values, rstds, q, base, coeffs, c0):
    """One read (b, t, d): base + sum_i (tc_i - coeffs_i) v_i and tc."""
    z = torch.stack([(v * q).sum(-1) for v in values], -1) * rstds / math.sqrt(q.shape[-1])
    lc = c0.clamp_min(1e-8).log()
    tc = c0 + c0.sum() * (torch.softmax(z + lc, -1) - torch.softmax(lc, -1))
    out = base
    for i, v in enumerate(values):
        out = out + (tc[..., i] - coeffs[..., i])[..., None] * v
    return out, tc


def _loop64(block, h0, Q, K, R, eps):
    """The layer loop with the read; block(k, s, x) is the s-th block application, of block k."""
    h, values, rstds, coeffs, c0 = h0, [], [], None, None
    lam = 1.0 - BETA
    for s in range(K * R):
        x = h
        hs = block(s % K, s, x)
        v = hs - x
        values.append(v)
        rstds.append(torch.rsqrt(v.pow(2).mean(-1) + eps))
        one = torch.ones_like(rstds[0])[..., None]
        coeffs = one if coeffs is None else torch.cat((coeffs, one), -1)
        c0 = one.new_ones(1) if c0 is None else torch.cat((c0, one.new_ones(1)))
        base = hs
        if s % K == K - 1:
            base, coeffs, c0 = hs + BETA * (h0 - hs), lam * coeffs, lam * c0
        if s == 0:
            h = base
        else:
            h, coeffs = _read64(values, torch.stack(rstds, -1), Q[s - 1], base, coeffs, c0)
    return h


def _chain_exact(case, seed):
    h0, D, Q, G = _chain_inputs(case, seed)
    train = case["kind"] == "train"
    d, T, N = case["d"], case["b"] * case["t"], case["K"] * case["R"]
    h0, D = h0.view(1, T, d), [x.view(1, T, d) for x in D]
    chunk = max(1, min(T, int(6e9 / (8 * d * N * N))))      # tokens are independent but for the query's gradient
    hs, gh0, gD, gQ = [], [], [[] for _ in D], torch.zeros(Q.shape, dtype=torch.float64, device=Q.device)
    with torch.set_grad_enabled(train):
        for t in range(0, T, chunk):
            a = h0[:, t:t + chunk].double().requires_grad_(train)
            ds = [x[:, t:t + chunk].double().requires_grad_(train) for x in D]
            q = Q.double().requires_grad_(train)
            h = _loop64(lambda k, s, x: x + ds[s], a, q, case["K"], case["R"], EPS)
            hs.append(h.detach())
            if train:
                (h * G.view(1, T, d)[:, t:t + chunk].double()).sum().backward()
                gh0.append(a.grad)
                gQ += q.grad
                for acc, x in zip(gD, ds):
                    acc.append(x.grad)
    shape = (case["b"], case["t"], d)
    cat = lambda xs: torch.cat(xs, 1).view(shape)
    return [cat(hs), cat(gh0), gQ, *[cat(x) for x in gD]] if train else cat(hs)


def _norm64(x, w):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + 1e-6) * w


def _block64(w, prefix, x, heads):
    """Pre-norm causal rotary attention and SwiGLU, one sequence (t, d) at a time."""
    t, d = x.shape
    dh = d // heads
    q, k, v = (_norm64(x, w[prefix + "attn_norm.weight"]) @ w[prefix + "attn.qkv.weight"].T).view(t, 3, heads, dh) \
        .permute(1, 2, 0, 3).unbind(0)
    ang = torch.outer(torch.arange(t, device=x.device, dtype=x.dtype),
                      1e6 ** (-torch.arange(0, dh, 2, device=x.device, dtype=x.dtype) / dh))
    cos, sin = torch.cat((ang.cos(), ang.cos()), -1), torch.cat((ang.sin(), ang.sin()), -1)
    turn = lambda y: y * cos + torch.cat((-y[..., dh // 2:], y[..., :dh // 2]), -1) * sin
    s = (turn(q) @ turn(k).transpose(1, 2).contiguous()) / math.sqrt(dh)
    s = s.masked_fill(torch.ones(t, t, dtype=torch.bool, device=x.device).triu(1), -math.inf)
    a = (torch.softmax(s, -1) @ v.contiguous()).transpose(0, 1).reshape(t, d)
    x = x + a @ w[prefix + "attn.o.weight"].T
    g, u = (_norm64(x, w[prefix + "mlp_norm.weight"]) @ w[prefix + "mlp.gate_up.weight"].T).chunk(2, -1)
    return x + (torch.nn.functional.silu(g) * u) @ w[prefix + "mlp.down.weight"].T


def _logits64(w, case, ids):
    H = case["heads"]
    h = w["embed.weight"][ids]
    for i in range(case["P"]):
        h = _block64(w, f"prelude.{i}.", h, H)
    h = _loop64(lambda k, s, x: _block64(w, f"middle.{k}.", x[0], H)[None], h[None], w["read.query"], case["K"],
                case["R"], 1e-6)[0]
    for i in range(case["C"]):
        h = _block64(w, f"coda.{i}.", h, H)
    return _norm64(h, w["norm.weight"]) @ w["head.weight"].T


def _lm_exact(case, seed):
    kind = case["kind"]
    train = kind != "prefill"
    w = {name: x.double().requires_grad_(train) for name, x in _weights(case, seed).items()}
    inputs = _lm_inputs(case, seed)
    outs, gx, loss = [], [], 0.0
    with torch.set_grad_enabled(train):
        for i in range(case["b"]):                            # one sequence at a time
            if kind == "block":
                x = inputs[0][i].double().requires_grad_()
                y = _block64(w, "", x, case["heads"])
                y.backward(inputs[1][i].double())
                outs.append(y.detach())
                gx.append(x.grad)
                continue
            logits = _logits64(w, case, inputs[i])
            if kind == "prefill":
                outs.append(logits)
                continue
            part = torch.nn.functional.cross_entropy(logits[:-1], inputs[i][1:], reduction="sum")
            part = part / (case["b"] * (case["t"] - 1))
            part.backward()
            loss = loss + part.detach()
    if kind == "prefill":
        return torch.stack(outs)
    grads = {name: x.grad for name, x in w.items()}
    return {"y": torch.stack(outs), "x": torch.stack(gx), **grads} if kind == "block" else {"loss": loss, **grads}


def exact(case: dict, seed: int):
    return (_chain_exact if case["kind"] in ("graph_eval", "eval", "train") else _lm_exact)(case, seed)
