"""The workloads that this framework's speed is judged on.

``listed()`` holds the cases themselves, ``draw(rng)`` makes more of the same ranges. A case is a
dict of plain values whose ``"kind"`` names the public entry point that it calls:

* ``decode``   ``WKV7Runner.decode_step``: one token for each of a batch of slots, every layer
* ``fla``      ``fused_recurrent_rwkv7`` / ``chunk_rwkv7``: the model layer's WKV op, from one
               token to whole prompts, dense or packed
* ``mixed``    ``WKV7Runner.mixed_step``: decode rows and ragged prompts in one scheduler step
* ``graph``    ``TimeMixDecodeGraph``: a decode step of whole time-mix blocks
* ``block``    ``RWKV7TimeMix.forward``: one time-mix block over packed prompts
* ``fork``     ``RWKV7StateBank.fork_slots``: every layer's state of some slots to fresh slots

Shapes are those of RWKV-7 0.1B (12 heads), 1.5B (32) and 7B (64); batch and prompt sizes are those
of the repository's benchmark and of a serving engine around them. Only as many layers as keep the
working set above the last-level cache are run: a layer's cost does not depend on how many follow.
"""

from __future__ import annotations

import math
import random

import torch

import wkvm_amd
from wkvm_amd import RWKV7StateBank, RWKV7StateLayout, WKV7Runner
from wkvm_amd.timemix import RWKV7TimeMix, TimeMixDecodeGraph, TokenBatch

DEV = "cuda"
N = 64  # head size
DECAY = 0.6065306597126334  # exp(-1/2): RWKV-7's log-decay is -DECAY * sigmoid(.)
SHAPES = {12: (12, 768), 32: (24, 2048), 64: (32, 4096)}  # heads -> (layers, hidden size)


def listed():
    return [
        # A small model with a handful of live requests: launches and host work are all there is.
        {"name": "decode_small", "kind": "decode", "heads": 12, "layers": 12, "slots": 16,
         "batch": 4, "f32": False},
        # The headline decode step: 256 live requests scattered over a 512-slot pool.
        {"name": "decode_256", "kind": "decode", "heads": 32, "layers": 4, "slots": 512,
         "batch": 256, "f32": False},
        # The model layer's op called for one token of each request (states held by a cache).
        {"name": "fla_step", "kind": "fla", "heads": 32, "seqs": 64, "tokens": 1, "ragged": False,
         "state": True},
        # A few short prompts packed into one call (below the 64 tokens where the model layer
        # switches to the chunked op).
        {"name": "fla_short", "kind": "fla", "heads": 32, "seqs": 5, "tokens": 63, "ragged": True,
         "state": True},
        # The engine's prefill: one request, one 512-token slice, continuing from its state.
        {"name": "chunk_slice", "kind": "fla", "heads": 32, "seqs": 1, "tokens": 512,
         "ragged": False, "state": True},
        # The benchmark's prefill: eight long prompts at once, from empty states.
        {"name": "chunk_batch", "kind": "fla", "heads": 32, "seqs": 8, "tokens": 4096,
         "ragged": False, "state": False},
        # One long document.
        {"name": "chunk_long", "kind": "fla", "heads": 32, "seqs": 1, "tokens": 16384,
         "ragged": False, "state": False},
        # A scheduler step of a busy engine: 448 decode rows beside 64 prompts of 1..2048 tokens.
        {"name": "mixed_step", "kind": "mixed", "heads": 32, "layers": 2, "slots": 1024,
         "batch": 448, "seqs": 64, "tokens": 2048},
        # A decode step of whole time-mix blocks at the headline batch, and at a few requests.
        {"name": "graph_256", "kind": "graph", "heads": 32, "layers": 4, "slots": 512,
         "batch": 256},
        {"name": "graph_8", "kind": "graph", "heads": 32, "layers": 4, "slots": 64, "batch": 8},
        # A time-mix block over a packed batch of prompts.
        {"name": "block_prefill", "kind": "block", "heads": 32, "slots": 16, "seqs": 4,
         "tokens": 1500},
        # Prefix sharing: a state forked to fresh slots in every layer.
        {"name": "fork_32", "kind": "fork", "heads": 32, "layers": 24, "slots": 96, "pairs": 32},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "fla", "fla", "fla", "mixed", "graph", "block", "block", "fork"])
    heads = rng.choice([12, 32, 32, 64])
    if kind == "decode":
        batch = _log(rng, 1, 448 * 32 // max(heads, 32))
        return {"kind": kind, "heads": heads, "layers": 4, "slots": batch + _log(rng, 1, 256),
                "batch": batch, "f32": rng.random() < 0.3}
    if kind == "fla":
        seqs = _log(rng, 1, 32)
        if rng.random() < 0.2:
            tokens = 1
            seqs = _log(rng, 1, 256)
        else:  # at most the listed batch's token-heads
            tokens = _log(rng, 2, min(16384, (1 << 20) // (seqs * heads)))
        return {"kind": kind, "heads": heads, "seqs": seqs, "tokens": tokens,
                "ragged": tokens > 1 and rng.random() < 0.6, "state": rng.random() < 0.6}
    if kind == "mixed":
        batch, seqs = _log(rng, 1, 224), _log(rng, 1, 32)
        return {"kind": kind, "heads": heads, "layers": 1, "slots": batch + seqs + 64,
                "batch": batch, "seqs": seqs, "tokens": _log(rng, 2, 2048)}
    if kind == "graph":
        batch = _log(rng, 1, 300)
        return {"kind": kind, "heads": rng.choice([12, 32, 32]), "layers": 3,
                "slots": batch + _log(rng, 1, 128), "batch": batch}
    if kind == "block":
        seqs = _log(rng, 1, 16)
        return {"kind": kind, "heads": rng.choice([12, 32, 32]), "slots": 32, "seqs": seqs,
                "tokens": _log(rng, 2, 8192 // seqs)}
    pairs = _log(rng, 1, 32)
    return {"kind": kind, "heads": heads, "layers": SHAPES[heads][0] * 32 // max(heads, 32),
            "slots": 2 * pairs + _log(rng, 1, 32), "pairs": pairs}


def _lengths(case):
    """Tokens of each prompt: uniform in 1..tokens where the batch is ragged, with the longest
    among them."""
    if case["kind"] == "fla" and not case["ragged"]:
        return [case["tokens"]] * case["seqs"]
    rng = random.Random("%(seqs)d prompts of at most %(tokens)d tokens" % case)
    lens = [rng.randint(1, case["tokens"]) for _ in range(case["seqs"])]
    lens[rng.randrange(len(lens))] = case["tokens"]
    return lens


def _cu(lens):
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    return cu


class _Rand:
    """Seeded values on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEV)
        self.g.manual_seed(int(seed))

    def normal(self, shape, std=1.0, dtype=torch.bfloat16):
        return (torch.randn(shape, generator=self.g, device=DEV) * std).to(dtype)

    def uniform(self, shape, lo, hi):
        return (torch.rand(shape, generator=self.g, device=DEV) * (hi - lo) + lo).bfloat16()

    def slots(self, count, total):
        """``count`` distinct slots of 1..total (row 0 is the pad slot)."""
        return (torch.randperm(total, generator=self.g, device=DEV)[:count] + 1).tolist()

    def vectors(self, *shape):
        """The WKV op's r, w, k, v, a, b as an RWKV-7 time-mix makes them: unit keys in a and b,
        a gate in (0, 1), log-decays in (-0.607, 0)."""
        shape = (*shape, N)
        r, k, v = (self.normal(shape) for _ in range(3))
        w = (-DECAY * torch.sigmoid(self.normal(shape).float())).bfloat16()
        kk = torch.nn.functional.normalize(k.float(), dim=-1)
        b = (kk * torch.sigmoid(self.normal(shape).float())).bfloat16()
        return r, w, k, v, (-kk).bfloat16(), b


def _layout(case, layers):
    hidden = case["heads"] * N
    return RWKV7StateLayout(n_layer=layers, hidden_size=hidden, num_heads=case["heads"],
                            head_dim=N, head_v_dim=N, dtype=torch.bfloat16)


def _bank(case, layers, rnd):
    """A pool in use: every slot holds a state."""
    bank = RWKV7StateBank(_layout(case, layers), case["slots"], DEV)
    bank.wkv.normal_(0.0, 0.1, generator=rnd.g)
    bank.shift.normal_(0.0, 1.0, generator=rnd.g)
    return bank


def _weights(hidden, layer, rnd):
    """A time-mix layer's parameters, [out, in], at a trained layer's scale of activations."""
    r32 = lambda x: max(32, int(round(x / 32)) * 32)  # noqa: E731
    ranks = {"w": r32(1.8 * hidden ** 0.5), "a": r32(1.8 * hidden ** 0.5),
             "v": r32(1.3 * hidden ** 0.5), "g": r32(0.6 * hidden ** 0.8)}
    W = {"mix": rnd.uniform((6, hidden), 0.0, 1.0)}
    for name in "rkvo":
        W[name] = rnd.normal((hidden, hidden), hidden ** -0.5)
    for name, rank in ranks.items():
        if name == "v" and layer == 0:
            continue
        W[name + "1"] = rnd.normal((rank, hidden), hidden ** -0.5)
        W[name + "2"] = rnd.normal((hidden, rank), rank ** -0.5)
        if name != "g":
            W[name + "0"] = rnd.normal((hidden,), 0.5)
    W["k_k"] = rnd.uniform((hidden,), 0.5, 1.5)
    W["k_a"] = rnd.uniform((hidden,), 0.0, 1.0)
    W["r_k"] = rnd.normal((hidden,), 0.1)
    W["ln_w"] = rnd.uniform((hidden,), 0.8, 1.2)
    W["ln_b"] = rnd.normal((hidden,), 0.05)
    return W


def _dicts(slots):
    """Slot ids as the engine's arena hands them out."""
    return [{"wkv": s, "shift": s} for s in slots]


def _inputs(case, seed):
    """Everything that prepare() and exact() have in common, from the seed alone."""
    rnd, kind = _Rand(seed), case["kind"]
    s = {"case": case}
    if kind == "fla":
        s["lens"] = _lengths(case)
        total = sum(s["lens"])
        lead = (1, total) if case["ragged"] else (case["seqs"], case["tokens"])
        s["x"] = rnd.vectors(*lead, case["heads"])
        s["h0"] = (rnd.normal((case["seqs"], case["heads"], N, N), 0.1, torch.float32)
                   if case["state"] else None)
        return s
    layers = case.get("layers", 1)
    # A block that needs v_first is the second of its model.
    s["bank"] = _bank(case, 2 if kind == "block" else layers, rnd)
    if kind == "decode":
        s["slots"] = rnd.slots(case["batch"], case["slots"])
        s["x"] = [rnd.vectors(case["batch"], case["heads"]) for _ in range(layers)]
    elif kind == "mixed":
        s["lens"] = _lengths(case)
        both = rnd.slots(case["batch"] + case["seqs"], case["slots"])
        s["slots"], s["prefill"] = both[:case["batch"]], both[case["batch"]:]
        s["x"] = [rnd.vectors(case["batch"], case["heads"]) for _ in range(layers)]
        s["px"] = [rnd.vectors(sum(s["lens"]), case["heads"]) for _ in range(layers)]
    elif kind == "graph":
        hidden = case["heads"] * N
        s["slots"] = rnd.slots(case["batch"], case["slots"])
        s["W"] = [_weights(hidden, layer, rnd) for layer in range(layers)]
        s["x"] = rnd.normal((layers, case["batch"], hidden))
    elif kind == "block":
        hidden = case["heads"] * N
        s["lens"] = _lengths(case)
        s["slots"] = rnd.slots(case["seqs"], case["slots"])
        s["W"] = _weights(hidden, 1, rnd)
        s["x"] = rnd.normal((sum(s["lens"]), hidden))
        s["v_first"] = rnd.normal((sum(s["lens"]), hidden))
    else:
        both = rnd.slots(2 * case["pairs"], case["slots"])
        s["src"], s["dst"] = both[:case["pairs"]], both[case["pairs"]:]
    return s


def prepare(case, seed):
    s = _inputs(case, seed)
    kind = case["kind"]
    if kind == "fla":
        # packed prompts come with the offsets on the device, as the model forward passes them
        s["cu"] = (torch.tensor(_cu(s["lens"]), dtype=torch.int64, device=DEV)
                   if case["ragged"] else None)
        # below 64 tokens the model layer takes the recurrent op
        s["op"] = (wkvm_amd.fused_recurrent_rwkv7 if case["tokens"] < 64
                   else wkvm_amd.chunk_rwkv7)
    elif kind in ("decode", "mixed"):
        s["runner"] = WKV7Runner(s["bank"])
        s["batch"] = _dicts(s["slots"])
        if kind == "mixed":
            s["pbatch"] = _dicts(s["prefill"])
    elif kind == "graph":
        bank = s["bank"]
        blocks = [RWKV7TimeMix(bank.layout, i, W) for i, W in enumerate(s["W"])]
        s["graph"] = TimeMixDecodeGraph(bank, blocks, case["batch"])
        s["graph"].x.copy_(s["x"])
    elif kind == "block":
        s["block"] = RWKV7TimeMix(s["bank"].layout, 1, s["W"])
        s["plan"] = TokenBatch.plan(s["bank"], s["slots"], _cu(s["lens"]))
    else:
        s["from"], s["to"] = _dicts(s["src"]), _dicts(s["dst"])
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "fla":
        return s["op"](*s["x"], initial_state=s["h0"], output_final_state=True,
                       cu_seqlens=s["cu"])
    bank = s["bank"]
    if kind == "decode":
        y = s["runner"].decode_step(s["batch"], s["x"],
                                    torch.float32 if case["f32"] else torch.bfloat16)
        return {"y": y, "wkv": bank.wkv}
    if kind == "mixed":
        y, py = s["runner"].mixed_step(s["batch"], s["x"], s["pbatch"], s["lens"], s["px"])
        return {"y": y, "py": py, "wkv": bank.wkv}
    if kind == "graph":
        s["graph"].set_slots(s["slots"])
        return {"y": s["graph"].replay(), "wkv": bank.wkv, "shift": bank.shift}
    if kind == "block":
        y, _ = s["block"].forward(bank, s["x"], s["plan"], s["v_first"])
        return {"y": y, "wkv": bank.wkv, "shift": bank.shift}
    bank.fork_slots(s["from"], s["to"])
    return {"wkv": bank.wkv, "shift": bank.shift}


def work(case):
    heads, kind = case["heads"], case["kind"]
    hidden = heads * N
    tile = 4 * N * N  # bytes of one head's state
    # A token of one head: six bf16 vectors in, one out; decay, p, two rank-one updates and y.
    token_b, token_f = 7 * 2 * N, 9 * N * N
    if kind == "fla":
        tokens = sum(_lengths(case)) * heads
        states = case["seqs"] * heads * (2 if case["state"] else 1)
        return {"bytes": tokens * token_b + states * tile, "flops": tokens * token_f}
    layers = case.get("layers", 1)
    if kind == "decode":
        rows = case["batch"] * heads * layers
        y = 2 * N if case["f32"] else 0
        return {"bytes": rows * (2 * tile + token_b + y), "flops": rows * token_f}
    if kind == "mixed":
        rows, tokens = case["batch"] * heads, sum(_lengths(case)) * heads
        return {"bytes": layers * (2 * tile * (rows + case["seqs"] * heads)
                                   + token_b * (rows + tokens)),
                "flops": layers * token_f * (rows + tokens)}
    if kind == "fork":
        row = heads * tile + 2 * 2 * hidden
        return {"bytes": 2 * case["pairs"] * layers * row, "flops": 0}
    # time-mix blocks: weights once, x in and the output out, states and shift rows both ways
    r32 = lambda x: max(32, int(round(x / 32)) * 32)  # noqa: E731
    ranks = 2 * r32(1.8 * hidden ** 0.5) + r32(1.3 * hidden ** 0.5) + r32(0.6 * hidden ** 0.8)
    weights = 4 * hidden * hidden + 2 * ranks * hidden
    if kind == "graph":
        rows, states = case["batch"], case["batch"]
    else:
        rows, states = sum(_lengths(case)), case["seqs"]
    nbytes = (2 * weights + 2 * 2 * rows * hidden + (2 * rows * hidden if kind == "block" else 0)
              + states * (2 * heads * tile + 2 * 2 * hidden))
    return {"bytes": layers * nbytes, "flops": layers * rows * (2 * weights + heads * token_f)}


def tolerance(case):
    if case["kind"] == "fork":
        return "exact"
    if case["kind"] in ("graph", "block"):
        # bf16 between the stages of a block
        return {"rel": 2e-2, "max": 0.5}
    # bf16 outputs (rounding alone: 1.7e-3), states held in fp32
    return {"rel": 7e-3, "max": 0.2}


# -- the same in 64 bits, without the framework ------------------------------------------


def _scan(x, lens, h, zero=False):
    """The recurrence token by token: ``x`` six ``[T, H, 64]``, ``h`` ``[n, H, 64 keys, 64
    values]`` in 64 bits. Returns ``(y, h)``."""
    order = sorted(range(len(lens)), key=lambda i: -lens[i])
    cu = _cu(lens)
    first = torch.tensor([cu[i] for i in order], device=DEV)
    r, w, k, v, a, b = (t.double() for t in x)
    w = w.exp()
    h = h[order].clone()
    y = torch.empty_like(r)
    live = len(order)
    for t in range(lens[order[0]] if order else 0):
        while lens[order[live - 1]] <= t:
            live -= 1
        at = first[:live] + t
        hs = h[:live]
        p = torch.matmul(a[at].unsqueeze(-2), hs)
        hs = hs * w[at].unsqueeze(-1) + b[at].unsqueeze(-1) * p
        hs += k[at].unsqueeze(-1) * v[at].unsqueeze(-2)
        h[:live] = hs
        y[at] = torch.matmul(r[at].unsqueeze(-2), hs).squeeze(-2)
    back = torch.empty_like(h)
    back[order] = h
    return y, back


def _block(W, x, prev, v_first, lens, h, heads):
    """One time-mix block: ``(out, v, states)``. ``prev`` is each token's predecessor."""
    W = {n: t.double() for n, t in W.items()}
    delta = prev - x
    xr, xw, xk, xv, xa, xg = (x + delta * W["mix"][i] for i in range(6))
    tokens = x.shape[0]
    split = lambda t: t.reshape(tokens, heads, N)  # noqa: E731
    r, k, v = xr @ W["r"].T, xk @ W["k"].T, xv @ W["v"].T
    w = -DECAY * torch.sigmoid(torch.tanh(xw @ W["w1"].T) @ W["w2"].T + W["w0"])
    gate = torch.sigmoid(xa @ W["a1"].T @ W["a2"].T + W["a0"])
    g = torch.sigmoid(xg @ W["g1"].T) @ W["g2"].T
    if "v1" in W:
        v = v + (v_first - v) * torch.sigmoid(xv @ W["v1"].T @ W["v2"].T + W["v0"])
    kk = torch.nn.functional.normalize(split(k * W["k_k"]), dim=-1)
    k = k * (1 + (gate - 1) * W["k_a"])
    r, k, w, vh, gate = split(r), split(k), split(w), split(v), split(gate)
    y, h = _scan((r, w, k, vh, -kk, kk * gate), lens, h)
    y = y - y.mean(-1, keepdim=True)
    y = y / torch.sqrt(y.square().mean(-1, keepdim=True) + N * 1e-5)
    y = y.reshape(tokens, -1) * W["ln_w"] + W["ln_b"]
    bonus = (r * k * split(W["r_k"].expand(tokens, -1))).sum(-1, keepdim=True) * vh
    return ((y + bonus.reshape(tokens, -1)) * g) @ W["o"].T, v, h


def exact(case, seed):
    s = _inputs(case, seed)
    kind, heads = case["kind"], case["heads"]
    if kind == "fla":
        lens = s["lens"]
        x = [t.reshape(-1, heads, N) for t in s["x"]]
        h = (s["h0"].double() if case["state"]
             else torch.zeros((len(lens), heads, N, N), dtype=torch.float64, device=DEV))
        y, h = _scan(x, lens, h)
        return y.reshape(s["x"][0].shape), h
    wkv, shift = s["bank"].wkv, s["bank"].shift
    if kind == "fork":
        wkv[:, s["dst"]] = wkv[:, s["src"]]
        shift[:, :, s["dst"]] = shift[:, :, s["src"]]
        return {"wkv": wkv.double(), "shift": shift.double()}
    out = {}
    if kind == "decode":
        ones, out["y"] = [1] * case["batch"], []
        wkv = wkv.double()
        for layer, x in enumerate(s["x"]):
            y, wkv[layer, s["slots"]] = _scan(x, ones, wkv[layer, s["slots"]])
            out["y"].append(y)
    elif kind == "mixed":
        ones, out["y"], out["py"] = [1] * case["batch"], [], []
        wkv = wkv.double()
        for layer, (x, px) in enumerate(zip(s["x"], s["px"])):
            y, wkv[layer, s["slots"]] = _scan(x, ones, wkv[layer, s["slots"]])
            py, wkv[layer, s["prefill"]] = _scan(px, s["lens"], wkv[layer, s["prefill"]])
            out["y"].append(y)
            out["py"].append(py)
    else:
        lens = s["lens"] if kind == "block" else [1] * case["batch"]
        cu, slots = _cu(lens), s["slots"]
        wkv, shift = wkv.double(), shift.double()
        first, last = cu[:-1], [c - 1 for c in cu[1:]]
        layers = [(1, s["W"], s["x"])] if kind == "block" else [
            (i, W, s["x"][i]) for i, W in enumerate(s["W"])]
        v_first = s["v_first"].double() if kind == "block" else None
        outs = []
        for layer, W, x in layers:
            x = x.double()
            prev = torch.roll(x, 1, 0)
            prev[first] = shift[layer, 0, slots]
            shift[layer, 0, slots] = x[last]
            y, v, wkv[layer, slots] = _block(W, x, prev, v_first, lens, wkv[layer, slots], heads)
            v_first = v if layer == 0 else v_first
            outs.append(y)
        out["y"] = outs[0] if kind == "block" else outs
        out["shift"] = shift
    out["wkv"] = wkv
    return out
