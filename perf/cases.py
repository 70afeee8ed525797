"""The framework's main path as cases to time: generation, prompt processing, training
chunks, and the layers and blocks they are made of, at the sizes of the benchmark's
workloads and of the tests.

Each kind of case calls public entry points the way train.py's and generate.py's loops
reach them. `exact` restates the same maths in plain torch at 64 bits.
"""
import math

import torch
import torch.nn.functional as F
from torch import nn

from gruboros_amd import blocks
from gruboros_amd.linear import feed_forward
from gruboros_amd.mingru.minGRU import minGRU
from gruboros_amd.mingru.minLM import FeedForward, minLM
from gruboros_amd.optim import AdamWScheduleFree
from gruboros_amd.scan import gate_scan

EPS = float(torch.finfo(torch.float32).eps)  # RMSNorm's eps
VOCAB = 256  # bytes
CAST = {"bf16": torch.bfloat16, "f32": torch.float32, "f16": torch.float16}


def listed():
    return [
        # generate.py's loop: one token a call at batch 1, the production run's widths, a
        # model cast to bf16. The smallest work: launches and latency.
        {"name": "generate b1 d1024 e3", "kind": "decode", "precision": "bf16", "dim": 1024, "expansion": 3.0,
         "ff_mult": 1.5, "depth": 12, "batch": 1, "tokens": 8},
        # generate.py's first call: the whole prompt in parallel, ragged length, logits of
        # every position.
        {"name": "prompt b1 t777 d1024 e3", "kind": "prompt", "precision": "bf16", "dim": 1024, "expansion": 3.0,
         "ff_mult": 1.5, "depth": 12, "batch": 1, "length": 777},
        # Two TBPTT chunks of the production run (batch 1, chunk 2048, hiddens carried, the
        # second chunk's gradients added to the first's), a few of its layers.
        {"name": "train chunks b1 t2048 d1024 e3", "kind": "train", "dim": 1024, "expansion": 3.0, "ff_mult": 1.5,
         "depth": 4, "batch": 1, "length": 2048, "chunks": 2},
        # One minGRU block, forward and backward, of the 8-layer benchmark model (batch 8,
        # 2048 bytes of which 2047 are predicted from) and of the production run.
        {"name": "gru block b8 t2047 d1024 e1", "kind": "gru", "dim": 1024, "expansion": 1.0, "batch": 8,
         "length": 2047, "carried": False},
        {"name": "gru block b1 t2048 d1024 e3", "kind": "gru", "dim": 1024, "expansion": 3.0, "batch": 1,
         "length": 2048, "carried": True},
        # One FeedForward block, forward and backward, of the same two models.
        {"name": "ff block b8 t2047 d1024 m4", "kind": "ff", "dim": 1024, "ff_mult": 4.0, "batch": 8, "length": 2047,
         "branch": False},
        {"name": "ff block b1 t2048 d1024 m1.5", "kind": "ff", "dim": 1024, "ff_mult": 1.5, "batch": 1,
         "length": 2048, "branch": True},
        # Final norm, logits, cross-entropy and their gradients: every training step's end.
        {"name": "loss head b8 t2047 d1024", "kind": "head", "dim": 1024, "batch": 8, "length": 2047},
        # The single layer of an unchanged fp32 train.py: minGRU, and its FeedForward.
        {"name": "gru fp32 b4 t1024 d512", "kind": "gru_f32", "dim": 512, "expansion": 1.0, "batch": 4, "length": 1024,
         "carried": False},
        {"name": "ff fp32 b4 t1024 d512", "kind": "ff_f32", "dim": 512, "ff_mult": 4.0, "batch": 4, "length": 1024},
        # The scan by itself over long sequences, forward and backward: the largest stream.
        {"name": "scan b16 t8192 d2048 bf16", "kind": "scan", "precision": "bf16", "batch": 16, "length": 8192,
         "width": 2048, "carried": False},
        # The optimizer's step over the parameters of four production layers, embedding and head.
        {"name": "optimizer d1024 e3 l4", "kind": "optim", "dim": 1024, "expansion": 3.0, "ff_mult": 1.5, "depth": 4},
    ]


def _between(rng, low, high, of=1):
    """A multiple of `of` in [low, high], spread over the logarithm."""
    v = math.exp(rng.uniform(math.log(low), math.log(high)))
    return int(min(high, max(low, round(v / of) * of)))


def _one(rng):
    kind = rng.choice(["decode", "prompt", "train", "gru", "gru", "ff", "ff", "head", "gru_f32", "ff_f32", "scan",
                       "optim"])
    # widths: multiples of 64 mostly, of 16 at times (int(dim * 1.5) stays a multiple of 8)
    dim = _between(rng, 256, 2048, rng.choice([16, 64, 64, 128]))
    widths = {"dim": dim, "expansion": rng.choice([1.0, 1.5, 2.0, 3.0]), "ff_mult": rng.choice([1.5, 2.0, 4.0])}
    batch = rng.choice([1, 1, 2, 3, 4, 8])
    if kind == "decode":
        return {"kind": kind, "precision": rng.choice(["bf16", "bf16", "f32", "f16"]), **widths,
                "depth": rng.randint(2, 12), "batch": rng.randint(1, 8), "tokens": rng.randint(3, 12)}
    if kind == "prompt":
        return {"kind": kind, "precision": rng.choice(["bf16", "bf16", "f32"]), **widths, "depth": rng.randint(2, 12),
                "batch": rng.choice([1, 1, 2, 4]), "length": _between(rng, 16, 2048)}
    if kind == "train":
        return {"kind": kind, **widths, "depth": rng.randint(1, 4), "batch": batch,
                "length": _between(rng, 128, 2048), "chunks": rng.choice([1, 2])}
    if kind == "optim":
        return {"kind": kind, **widths, "depth": rng.randint(1, 4)}
    if kind == "scan":
        return {"kind": kind, "precision": rng.choice(["bf16", "bf16", "f32"]), "batch": rng.randint(1, 16),
                "length": _between(rng, 256, 16384), "width": _between(rng, 256, 4096, 8), "carried": rng.random() < 0.5}
    length = _between(rng, 128, 4096)
    if kind == "head":
        return {"kind": kind, "dim": dim, "batch": batch, "length": length}
    if kind in ("ff", "ff_f32"):
        case = {"kind": kind, "dim": dim, "ff_mult": widths["ff_mult"], "batch": batch, "length": length}
        return {**case, "branch": rng.random() < 0.5} if kind == "ff" else case
    return {"kind": kind, "dim": dim, "expansion": widths["expansion"], "batch": batch, "length": length,
            "carried": rng.random() < 0.5}


def _cost(case):
    w = work(case)
    return max(w["bytes"] / 6e12, w["flops"] / 1.2e15)


def draw(rng):
    """One more case of the listed kinds, at most as large as the largest listed one of its kind."""
    while True:
        case = _one(rng)
        if _cost(case) <= max(_cost(c) for c in listed() if c["kind"] == case["kind"]):
            return case


# ---------------------------------------------------------------------------- inputs


class _Draws:
    """Seeded normal tensors on the GPU."""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda").manual_seed(seed)

    def normal(self, *shape, std=1.0, mean=0.0, dtype=torch.float32):
        return torch.randn(*shape, generator=self.gen, device="cuda").mul_(std).add_(mean).to(dtype)

    def bytes(self, batch, length):
        """Byte ids as text has them: a few frequent ones, many rare."""
        u = torch.rand(batch, length, generator=self.gen, device="cuda", dtype=torch.float64)
        return ((VOCAB - 1) * u ** 3).long()

    def state(self, batch, width):
        """A recurrence state: positive, of order one."""
        return self.normal(batch, 1, width).abs_().add_(0.1)

    @torch.no_grad()
    def fill(self, module):
        """Weights as training leaves them: activations of order one, no zero blocks."""
        for name, p in module.named_parameters():
            if p.dim() == 1:
                p.copy_(self.normal(*p.shape, std=0.1, mean=0.0 if name.endswith("bias") else 1.0))
            elif name.startswith("token_emb"):
                p.copy_(self.normal(*p.shape, std=0.5))
            else:
                p.copy_(self.normal(*p.shape, std=0.7 / math.sqrt(p.shape[1])))
        return module


def _model(case, d, compute_dtype=None):
    with torch.device("cuda"):
        m = minLM(num_tokens=VOCAB, dim=case["dim"], depth=case["depth"], ff_mult=case["ff_mult"],
                  expansion=case["expansion"], compute_dtype=compute_dtype)
    return d.fill(m)


def _leaf(t):
    return t.requires_grad_(True)


def prepare(case, seed):
    d, kind = _Draws(seed), case["kind"]
    if kind in ("decode", "prompt"):
        model = _model(case, d).to(CAST[case["precision"]]).eval()
        s = {"kind": kind, "model": model}
        if kind == "prompt":
            return {**s, "ids": d.bytes(case["batch"], case["length"])}
        ids = d.bytes(case["batch"], case["tokens"])
        hiddens = [d.state(case["batch"], int(case["dim"] * case["expansion"])) for _ in range(case["depth"])]
        with torch.no_grad():  # a token generated before: what the loop keeps is there
            model(ids[:, :1], return_prev_hiddens=True, prev_hiddens=hiddens)
        return {**s, "ids": ids, "hiddens": hiddens}
    if kind == "train":
        model = _model(case, d, torch.bfloat16)
        return {"kind": kind, "model": model, "params": list(model.parameters()),
                "ids": [d.bytes(case["batch"], case["length"] + 1) for _ in range(case["chunks"])]}
    if kind == "optim":
        model = _model(case, d, torch.bfloat16)
        opt = AdamWScheduleFree(model.parameters(), lr=1e-3, betas=(0.9, 0.999), weight_decay=0.01)
        opt.train()
        with torch.no_grad():  # the 16-bit copies that training keeps beside the weights are there
            model(d.bytes(1, 17), return_loss=True)
        for p in model.parameters():
            p.grad = d.normal(*p.shape, std=1e-3)
        return {"kind": kind, "model": model, "opt": opt, "params": list(model.parameters())}
    if kind == "scan":
        shape, dtype = (case["batch"], case["length"], case["width"]), CAST[case["precision"]]
        hidden, gate = (_leaf(d.normal(*shape, dtype=dtype)) for _ in range(2))
        h0 = _leaf(d.state(case["batch"], case["width"])) if case["carried"] else None
        return {"kind": kind, "hidden": hidden, "gate": gate, "h0": h0, "dh": d.normal(*shape, std=1e-2, dtype=dtype)}
    B, T, D = case["batch"], case["length"], case["dim"]
    if kind == "gru_f32":
        with torch.device("cuda"):
            layer = minGRU(D, expansion_factor=case["expansion"])
        d.fill(layer)
        h0 = d.state(B, int(D * case["expansion"])) if case["carried"] else None
        return {"kind": kind, "layer": layer, "x": _leaf(d.normal(B, T, D)), "h0": h0,
                "dout": d.normal(B, T, D, std=1e-2)}
    if kind == "ff_f32":
        with torch.device("cuda"):
            layer = FeedForward(D, mult=case["ff_mult"])
        d.fill(layer)
        return {"kind": kind, "layer": layer, "x": _leaf(d.normal(B, T, D)), "dout": d.normal(B, T, D, std=1e-2)}
    with torch.device("cuda"):
        norm = nn.RMSNorm(D)
    d.fill(norm)
    x = _leaf(d.normal(B, T, D))
    s = {"kind": kind, "norm": norm, "x": x}
    if kind == "gru":
        with torch.device("cuda"):
            layer = minGRU(D, expansion_factor=case["expansion"])
        d.fill(layer)
        s.update(layer=layer, pending=_leaf(d.normal(B, T, D, std=0.3, dtype=torch.bfloat16)),
                 h0=d.state(B, int(D * case["expansion"])) if case["carried"] else None,
                 dx=d.normal(B, T, D, std=1e-2),
                 dout=d.normal(B, T, D, std=1e-2) if case["expansion"] != 1.0 else None)
    elif kind == "ff":
        with torch.device("cuda"):
            layer = FeedForward(D, mult=case["ff_mult"])
        d.fill(layer)
        s.update(layer=layer, branch=_leaf(d.normal(B, T, D)) if case["branch"] else None,
                 dx=d.normal(B, T, D, std=1e-2), dout=d.normal(B, T, D, std=1e-2, dtype=torch.bfloat16))
    else:  # head
        with torch.device("cuda"):
            layer = nn.Linear(D, VOCAB, bias=False)
        d.fill(layer)
        s.update(layer=layer, pending=_leaf(d.normal(B, T, D, std=0.3, dtype=torch.bfloat16)), labels=d.bytes(B, T))
    return s


# ---------------------------------------------------------------------------- the passes


def _clear(*tensors):
    for t in tensors:
        if t is not None:
            t.grad = None


def run(s):
    kind = s["kind"]
    if kind == "decode":
        model, hiddens, logits = s["model"], s["hiddens"], []
        with torch.no_grad():
            for i in range(s["ids"].shape[1]):
                out, hiddens = model(s["ids"][:, i:i + 1], return_prev_hiddens=True, prev_hiddens=hiddens)
                logits.append(out)
        return {"logits": logits, "hiddens": hiddens}
    if kind == "prompt":
        with torch.no_grad():
            logits, hiddens = s["model"](s["ids"], return_prev_hiddens=True)
        return {"logits": logits, "hiddens": hiddens}
    if kind == "train":
        _clear(*s["params"])
        hiddens, losses = None, []
        for ids in s["ids"]:
            loss, hiddens = s["model"](ids, return_loss=True, return_prev_hiddens=True, prev_hiddens=hiddens)
            hiddens = [h.detach() for h in hiddens]
            (loss / len(s["ids"])).backward()
            losses.append(loss.detach())
        return {"loss": losses, "hiddens": hiddens, "grads": [p.grad for p in s["params"]]}
    if kind == "optim":
        s["opt"].step()
        state = s["opt"].state
        return {"p": [p.detach() for p in s["params"]], "z": [state[p]["z"] for p in s["params"][:6]],
                "v": [state[p]["exp_avg_sq"] for p in s["params"][:6]]}
    if kind == "scan":
        hidden, gate, h0 = s["hidden"], s["gate"], s["h0"]
        _clear(hidden, gate, h0)
        h, last = gate_scan(hidden, gate, h0)
        h.backward(s["dh"])
        return {"h": h.detach(), "last": last.detach(), "dhidden": hidden.grad, "dgate": gate.grad,
                "dh0": h0.grad if h0 is not None else None}
    x, layer = s["x"], s["layer"]
    params = list(layer.parameters())
    _clear(x, *params)
    if kind == "gru_f32":
        out, last = layer(x, s["h0"], return_next_prev_hidden=True)
        out.backward(s["dout"])
        return {"out": out.detach(), "last": last.detach(), "dx": x.grad, "grads": [p.grad for p in params]}
    if kind == "ff_f32":
        out = feed_forward(x, layer)
        out.backward(s["dout"])
        return {"out": out.detach(), "dx": x.grad, "grads": [p.grad for p in params]}
    norm = s["norm"]
    _clear(norm.weight)
    if kind == "gru":
        pending = s["pending"]
        _clear(pending)
        to_out = layer.to_out.weight if isinstance(layer.to_out, nn.Linear) else None
        nxt, out, last = blocks.MinGRUBlock.apply(x, pending, norm.weight, layer.to_hidden_and_gate.weight, s["h0"],
                                                  to_out)
        if out is None:
            nxt.backward(s["dx"])
        else:
            torch.autograd.backward([nxt, out], [s["dx"], s["dout"]])
        return {"x": nxt.detach(), "out": out.detach() if out is not None else None, "last": last.detach(),
                "dx": x.grad, "dpending": pending.grad, "grads": [norm.weight.grad] + [p.grad for p in params]}
    if kind == "ff":
        branch = s["branch"]
        _clear(branch)
        l1, l2 = layer[0], layer[2]
        nxt, out = blocks.FFBlock.apply(x, branch, norm.weight, l1.weight, l1.bias, l2.weight, l2.bias)
        torch.autograd.backward([nxt, out], [s["dx"], s["dout"]])
        return {"x": nxt.detach(), "out": out.detach(), "dx": x.grad,
                "dbranch": branch.grad if branch is not None else None,
                "grads": [norm.weight.grad] + [p.grad for p in params]}
    pending = s["pending"]
    _clear(pending)
    loss = blocks.FinalNormCE.apply(x, pending, norm.weight, layer.weight, s["labels"])
    loss.backward()
    return {"loss": loss.detach(), "dx": x.grad, "dpending": pending.grad, "grads": [norm.weight.grad, layer.weight.grad]}


# ---------------------------------------------------------------------------- least work


def _layer_weights(case):
    D = case["dim"]
    Di, Fw = int(D * case["expansion"]), int(D * case["ff_mult"])
    return 2 * Di * D + (Di * D if Di != D else 0) + 2 * Fw * D


def work(case):
    """Bytes: each input read and each output written once at the types the entry point takes and
    gives. Flops: the products' multiply-adds as 2."""
    kind = case["kind"]
    if kind in ("decode", "prompt"):
        size = 4 if case["precision"] == "f32" else 2
        n = case["depth"] * _layer_weights(case) + VOCAB * case["dim"]
        hid = 8 * case["depth"] * case["batch"] * int(case["dim"] * case["expansion"])
        calls, rows = (case["tokens"], 1) if kind == "decode" else (1, case["length"])
        rows *= case["batch"]
        return {"bytes": calls * (size * (n + rows * VOCAB) + hid), "flops": 2 * calls * rows * n}
    if kind in ("train", "optim"):
        n = case["depth"] * _layer_weights(case) + VOCAB * case["dim"]
        if kind == "optim":  # p, g, z, v in; p, z, v and the 16-bit copies out
            return {"bytes": 30 * (n + VOCAB * case["dim"]), "flops": 0}
        rows = case["batch"] * case["length"] * case["chunks"]
        return {"bytes": case["chunks"] * 12 * n, "flops": 6 * rows * n}
    if kind == "scan":
        n = case["batch"] * case["length"] * case["width"]
        return {"bytes": 9 * n * (2 if case["precision"] == "bf16" else 4), "flops": 0}
    D, N = case["dim"], case["batch"] * case["length"]
    if kind in ("gru", "gru_f32"):
        Di = int(D * case["expansion"])
        n = 2 * Di * D + (Di * D if Di != D else 0)
        # x, dout in and out, dx out; the block: x, pending, dx, dout in; x, out, dx, dpending out
        per = 16 if kind == "gru_f32" else 20 + (8 if Di != D else 0)
        return {"bytes": per * N * D + 8 * n, "flops": 6 * N * n}
    if kind in ("ff", "ff_f32"):
        n = 2 * int(D * case["ff_mult"]) * D
        per = 16 if kind == "ff_f32" else 20 + (8 if case["branch"] else 0)
        return {"bytes": per * N * D + 8 * n, "flops": 6 * N * n}
    return {"bytes": 12 * N * D + 8 * VOCAB * D + 8 * N, "flops": 6 * N * VOCAB * D}


# About four times the error against `exact`: 16-bit activations and stochastically rounded
# 16-bit gradients leave 3e-3 to 5e-3 in a block and up to 1e-2 over four layers' gradients,
# 16-bit logits 4e-3, 32-bit sums 2e-7 to 2e-6. A recurrent layer's gradient jumps where a
# pre-activation lands on the other side of the kink of g at 0: by the gradient's own size at
# that element, and, over the few million pre-activations of a 32-bit layer, by 4e-4 of the
# whole for a single one.
TOLERANCE = {"decode": 1.6e-2, "prompt": 1.6e-2, "train": 2.5e-2, "gru": 2e-2, "ff": 2e-2, "head": 1.6e-2,
             "gru_f32": 1e-3, "ff_f32": 8e-6, "scan": 1e-2, "optim": 3e-7}


def tolerance(case):
    kind = case["kind"]
    rel = TOLERANCE[kind]
    if case.get("precision") == "f32":
        rel = 2e-6
    return {"rel": rel, "max": 0.9 if kind in ("train", "gru", "gru_f32") else 40 * rel}


# ---------------------------------------------------------------------------- 64 bits


class _Recurrence(torch.autograd.Function):
    """h_t = a_t h_{t-1} + v_t over the first axis, one step after the other."""

    @staticmethod
    def forward(ctx, a, v, h0):
        h, prev = torch.empty_like(v), h0
        for t in range(v.shape[0]):
            prev = torch.addcmul(v[t], a[t], prev, out=h[t])
        ctx.save_for_backward(a, h, h0)
        return h

    @staticmethod
    def backward(ctx, dh):
        a, h, h0 = ctx.saved_tensors
        lam = dh.contiguous().clone()
        for t in range(lam.shape[0] - 2, -1, -1):
            lam[t].addcmul_(a[t + 1], lam[t + 1])
        da = torch.empty_like(a)
        torch.mul(lam[1:], h[:-1], out=da[1:])
        torch.mul(lam[0], h0, out=da[0])
        return da, lam, a[0] * lam[0]


def _g(x):
    return torch.where(x >= 0, torch.relu(x) + 0.5, torch.sigmoid(x))  # slope 0 at 0, as log(relu(x) + 0.5) has


def _scan64(hidden, gate, h0):
    """(h, last state) of [B, T, D] pre-activations and a [B, 1, D] state or None."""
    hidden, gate = hidden.transpose(0, 1).contiguous(), gate.transpose(0, 1).contiguous()
    first = h0[:, 0] if h0 is not None else torch.zeros_like(hidden[0])
    h = _Recurrence.apply(torch.sigmoid(-gate), torch.sigmoid(gate) * _g(hidden), first).transpose(0, 1)
    return h, h[:, -1:]


def _norm64(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w


def _gru64(x, w_hg, w_out, h0):
    hidden, gate = F.linear(x, w_hg).chunk(2, dim=-1)
    h, last = _scan64(hidden, gate, h0)
    return (F.linear(h, w_out) if w_out is not None else h), last


def _ff64(x, w1, b1, w2, b2):
    return F.linear(F.gelu(F.linear(x, w1, b1)), w2, b2)


def _model64(model, ids, hiddens):
    """Logits of every position and the next hiddens, from the model's parameters at 64 bits."""
    p = model["p"]
    x, following = F.embedding(ids, p["token_emb.weight"]), []
    for i in range(model["depth"]):
        q = {k[len("layers.%d." % i):]: v for k, v in p.items() if k.startswith("layers.%d." % i)}
        out, last = _gru64(_norm64(x, q["1.weight"]), q["2.to_hidden_and_gate.weight"], q.get("2.to_out.weight"),
                           hiddens[i] if hiddens is not None else None)
        following.append(last)
        x = x + out
        x = x + _ff64(_norm64(x, q["3.weight"]), q["4.0.weight"], q["4.0.bias"], q["4.2.weight"], q["4.2.bias"])
    return F.linear(_norm64(x, p["norm.weight"]), p["to_logits.weight"]), following


def _double(t, grad=False):
    return None if t is None else t.detach().double().requires_grad_(grad)


def exact(case, seed):
    kind = case["kind"]
    s = prepare(case, seed)
    if kind in ("decode", "prompt", "train"):
        train = kind == "train"
        named = {k: _double(v, train) for k, v in s["model"].named_parameters()}
        m = {"p": named, "depth": case["depth"]}
        if kind == "train":
            hiddens, losses = None, []
            for ids in s["ids"]:
                logits, hiddens = _model64(m, ids[:, :-1], hiddens)
                hiddens = [h.detach() for h in hiddens]
                loss = F.cross_entropy(logits.reshape(-1, VOCAB), ids[:, 1:].reshape(-1))
                (loss / len(s["ids"])).backward()
                losses.append(loss.detach())
            return {"loss": losses, "hiddens": hiddens, "grads": [v.grad for v in named.values()]}
        with torch.no_grad():
            if kind == "prompt":
                logits, hiddens = _model64(m, s["ids"], None)
                return {"logits": logits, "hiddens": hiddens}
            hiddens, rows = [_double(h) for h in s["hiddens"]], []
            for i in range(s["ids"].shape[1]):
                out, hiddens = _model64(m, s["ids"][:, i:i + 1], hiddens)
                rows.append(out)
            return {"logits": rows, "hiddens": hiddens}
    if kind == "optim":
        ps, zs, vs = [], [], []
        for p in s["params"]:  # the first step: z = p, v = 0, and the average's weight is all on z
            y, g = _double(p), _double(p.grad)
            v = 0.001 * g * g
            u = g / ((v / 0.001).sqrt() + 1e-8) + 0.01 * y
            ps.append(y - 1e-3 * u)
            zs.append(y - 1e-3 * u)
            vs.append(v)
        return {"p": ps, "z": zs[:6], "v": vs[:6]}
    if kind == "scan":
        hidden, gate, h0 = _double(s["hidden"], True), _double(s["gate"], True), _double(s["h0"], True)
        h, last = _scan64(hidden, gate, h0)
        h.backward(s["dh"].double())
        return {"h": h.detach(), "last": last.detach(), "dhidden": hidden.grad, "dgate": gate.grad,
                "dh0": h0.grad if h0 is not None else None}
    x = _double(s["x"], True)
    params = [_double(p, True) for p in s["layer"].parameters()]
    if kind in ("gru_f32", "gru"):
        w_hg, w_out = params[0], params[1] if len(params) > 1 else None
        h0 = _double(s["h0"])
    if kind == "gru_f32":
        out, last = _gru64(x, w_hg, w_out, h0)
        out.backward(s["dout"].double())
        return {"out": out.detach(), "last": last.detach(), "dx": x.grad, "grads": [p.grad for p in params]}
    if kind == "ff_f32":
        out = _ff64(x, *params)
        out.backward(s["dout"].double())
        return {"out": out.detach(), "dx": x.grad, "grads": [p.grad for p in params]}
    w = _double(s["norm"].weight, True)
    if kind == "gru":
        pending = _double(s["pending"], True)
        x1 = x + pending
        out, last = _gru64(_norm64(x1, w), w_hg, w_out, h0)
        if w_out is None:
            nxt, out = x1 + out, None
            nxt.backward(s["dx"].double())
        else:
            nxt = x1
            torch.autograd.backward([nxt, out], [s["dx"].double(), s["dout"].double()])
            out = out.detach()
        return {"x": nxt.detach(), "out": out, "last": last.detach(), "dx": x.grad, "dpending": pending.grad,
                "grads": [w.grad] + [p.grad for p in params]}
    if kind == "ff":
        branch = _double(s["branch"], True)
        x2 = x + branch if branch is not None else x * 1.0
        out = _ff64(_norm64(x2, w), *params)
        torch.autograd.backward([x2, out], [s["dx"].double(), s["dout"].double()])
        return {"x": x2.detach(), "out": out.detach(), "dx": x.grad, "dbranch": branch.grad if branch is not None else None,
                "grads": [w.grad] + [p.grad for p in params]}
    pending = _double(s["pending"], True)
    logits = F.linear(_norm64(x + pending, w), params[0])
    loss = F.cross_entropy(logits.reshape(-1, VOCAB), s["labels"].reshape(-1))
    loss.backward()
    return {"loss": loss.detach(), "dx": x.grad, "dpending": pending.grad, "grads": [w.grad, params[0].grad]}
