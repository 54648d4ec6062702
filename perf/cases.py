"""The work that programs have this library do, as measured cases.

listed() names the cases, draw() gives more of the same ranges, prepare() makes what a program
holds before the call (weights, pointer tables, scratch buffers, a captured step), run() is one
pass through the public entry points, exact() the same result in float64 from plain torch.

Four kinds of case:
  linear  one quantized linear layer (LinearEXL3): decode rows, small batches, prompt chunks
  qkv     q / k / v of one layer as one sliced bundle (bundles.Sliced)
  step    the linear part of a whole decode step, captured (DecodeStack)
  moe     routed experts with mixed bitrates: exl3_moe_coop for decode batches, exl3_moe for prompts

Weights: uniform random trellis words, which is how trained trellises look to the decoder;
suh / svh are signs with a spread of magnitudes, scaled so that a unit-variance input gives a
unit-variance output, as checkpoints carry them.  Activations: N(0, 1) fp16, what a norm emits.
"""
import math

import torch

from ampstein_amd import bundles, ops
from ampstein_amd.decode import DecodeStack, LayerWeights
from ampstein_amd.linear import LinearEXL3

DEV = "cuda"
CODEBOOKS = ("3inst", "mcg", "mul1")


# ------------------------------------------------------------------ cases
def listed():
    return [
        # one token through one projection of a small-hidden model: launch and latency count
        dict(name="row1_4096x4096_k4", kind="linear", rows=1, k=4096, n=4096, K=4.0, cb="3inst", bias=False),
        # q / k / v of four sequences (or a four-token draft) as one launch
        dict(name="qkv4_5120_k4", kind="qkv", rows=4, k=5120, n=5120, kv=1024, K=4.0, cb="3inst"),
        # a verify batch of 1 + 7 draft tokens through a wide FFN projection
        dict(name="verify8_5120x17408_k3", kind="linear", rows=8, k=5120, n=17408, K=3.0, cb="mcg", bias=False),
        # continuous batching: an odd number of sequences, one token each, through the FFN's way back
        dict(name="batch33_17408x5120_k4", kind="linear", rows=33, k=17408, n=5120, K=4.0, cb="3inst", bias=False),
        # a larger serving batch (or a short prompt), layer with a bias
        dict(name="batch100_4096x14336_k5", kind="linear", rows=100, k=4096, n=14336, K=5.0, cb="mul1", bias=True),
        # a ragged prompt chunk at a half-integer bitrate
        dict(name="chunk509_14336x4096_k3.5", kind="linear", rows=509, k=14336, n=4096, K=3.5, cb="mul1", bias=False),
        # a long prompt through the widest layer
        dict(name="prompt2048_8192x28672_k4", kind="linear", rows=2048, k=8192, n=28672, K=4.0, cb="3inst", bias=False),
        # the vocabulary head for one token: a very wide matrix at a high bitrate
        dict(name="head1_4096x128256_k6", kind="linear", rows=1, k=4096, n=128256, K=6.0, cb="mul1", bias=False),
        # a whole decode step of an 8B-class stack: 32 layers, one captured graph
        dict(name="step32_4096_k4", kind="step", layers=32, hidden=4096, kv=1024, inter=14336, K=4.0, cb="3inst"),
        # routed experts for a single token, a decode batch, and a prompt
        dict(name="moe1_256x4096x2048", kind="moe", tokens=1, experts=256, hidden=4096, inter=2048, topk=8),
        dict(name="moe16_256x4096x2048", kind="moe", tokens=16, experts=256, hidden=4096, inter=2048, topk=8),
        dict(name="moe1024_256x4096x2048", kind="moe", tokens=1024, experts=256, hidden=4096, inter=2048, topk=8),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _rate(rng):
    """A bitrate and a codebook it exists in (half-integer rates are mul1 only)."""
    cb = rng.choice(CODEBOOKS)
    K = rng.choice((2.0, 3.0, 4.0, 4.0, 5.0, 6.0, 8.0) + ((1.5, 2.5, 3.5) if cb == "mul1" else ()))
    return K, cb


def draw(rng):
    kind = rng.choice(("linear", "linear", "linear", "linear", "qkv", "step", "moe", "moe"))
    K, cb = _rate(rng)
    if kind == "linear":
        k, n = 128 * _log_int(rng, 8, 224), 128 * _log_int(rng, 8, 224)
        rows = min(_log_int(rng, 1, 3000), int(2048 * 8192 * 28672 / (k * n)))
        return dict(kind=kind, rows=rows, k=k, n=n, K=K, cb=cb, bias=rng.random() < 0.25)
    if kind == "qkv":
        k = 128 * rng.randint(8, 64)
        return dict(kind=kind, rows=_log_int(rng, 1, 16), k=k, n=k, kv=128 * rng.choice((2, 4, 8, 16)), K=K, cb=cb)
    if kind == "step":
        hidden = 128 * rng.randint(8, 40)
        return dict(kind=kind, layers=rng.randint(2, 24), hidden=hidden, kv=128 * rng.choice((2, 4, 8)),
                    inter=128 * rng.randint(16, 112), K=min(K, 4.0), cb=cb)
    return dict(kind=kind, tokens=_log_int(rng, 1, 16) if rng.random() < 0.6 else _log_int(rng, 64, 1024),
                experts=rng.choice((16, 64, 128, 256)), hidden=128 * rng.randint(8, 32), inter=128 * rng.randint(4, 16),
                topk=rng.choice((2, 4, 8)))


# ------------------------------------------------------------------ inputs
class _Store:
    """The weight store of a program that keeps its tensors on the device (the interface that
    LinearEXL3 reads a checkpoint through)."""

    def __init__(self, tensors):
        self.t = tensors

    def has(self, key):
        return key in self.t

    def info(self, key):
        return {"shape": list(self.t[key].shape)}

    def gpu(self, key, dev=None):
        return self.t[key]

    gpu16 = gpu


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _normal(g, *shape):
    return torch.randn(shape, generator=g, device=DEV, dtype=torch.float32).half()


def _scales(g, n, size):
    """n random signs times magnitudes spread by half around `size`."""
    sign = torch.randint(0, 2, (n,), generator=g, device=DEV) * 2 - 1
    return (sign * size * (0.75 + 0.5 * torch.rand(n, generator=g, device=DEV))).half()


def _matrix(g, k, n, K):
    """(trellis, suh, svh) of one k -> n layer."""
    t = torch.randint(-32768, 32768, (k // 16, n // 16, int(16 * K)), generator=g, device=DEV, dtype=torch.int16)
    return t, _scales(g, k, 1.0), _scales(g, n, 1.0 / math.sqrt(k))


def _linear_inputs(case, seed):
    g = _gen(seed)
    w = _matrix(g, case["k"], case["n"], case["K"])
    bias = _normal(g, case["n"]) if case["bias"] else None
    return w, bias, _normal(g, case["rows"], case["k"])


def _qkv_inputs(case, seed):
    g = _gen(seed)
    return ([_matrix(g, case["k"], n, case["K"]) for n in (case["n"], case["kv"], case["kv"])],
            _normal(g, 1, case["rows"], case["k"]))


def _step_inputs(case, seed):
    g = _gen(seed)
    H, V, I, K = case["hidden"], case["kv"], case["inter"], case["K"]
    shapes = dict(q=(H, H), k=(H, V), v=(H, V), o=(H, H), gate=(H, I), up=(H, I), down=(I, H))
    norm = lambda: (1.0 + 0.2 * torch.randn(H, generator=g, device=DEV)).half()
    layers = [({name: _matrix(g, *s, K) for name, s in shapes.items()}, norm(), norm()) for _ in range(case["layers"])]
    return layers, norm(), _normal(g, 1, H)


def _expert_K(case):
    return [2 + e % 3 for e in range(case["experts"])]


def _moe_inputs(case, seed):
    """Experts (gate, up, down), hidden rows, router choice and softmax weights."""
    g = _gen(seed)
    H, I, E = case["hidden"], case["inter"], case["experts"]
    experts = [[_matrix(g, H, I, K), _matrix(g, H, I, K), _matrix(g, I, H, K)] for K in _expert_K(case)]
    p, sel = torch.topk(torch.softmax(torch.randn(case["tokens"], E, generator=g, device=DEV), 1), case["topk"], dim=1)
    return experts, _normal(g, case["tokens"], H), sel.contiguous(), p.half().contiguous()


def _flags(case):
    return case["cb"] == "mcg", case["cb"] == "mul1"


def prepare(case, seed):
    return {"linear": _prepare_linear, "qkv": _prepare_qkv, "step": _prepare_step, "moe": _prepare_moe}[case["kind"]](case, seed)


def _prepare_linear(case, seed):
    (t, suh, svh), bias, x = _linear_inputs(case, seed)
    store = {"w.trellis": t, "w.suh": suh, "w.svh": svh}
    if case["cb"] != "3inst":
        store["w." + case["cb"]] = torch.zeros(1, dtype=torch.int8, device=DEV)
    if bias is not None:
        store["w.bias"] = bias
    return {"kind": "linear", "layer": LinearEXL3(_Store(store), "w"), "x": x}


def _prepare_qkv(case, seed):
    mats, x = _qkv_inputs(case, seed)
    lins = [bundles.Linear(*m, case["K"], *_flags(case)) for m in mats]
    outs = [torch.zeros((1, case["rows"], w.out_features), dtype=torch.half, device=DEV) for w in lins]
    return {"kind": "qkv", "bundle": bundles.Sliced(lins, outs), "keep": lins, "x": x}


def _prepare_step(case, seed):
    layers, final, x = _step_inputs(case, seed)
    lin = lambda m: bundles.Linear(*m, case["K"], *_flags(case))
    stack = DecodeStack([LayerWeights(**{nm: lin(m) for nm, m in mats.items()}, input_norm=a, post_norm=b)
                         for mats, a, b in layers], final)
    stack.capture()
    return {"kind": "step", "stack": stack, "x": x}


def _prepare_moe(case, seed):
    experts, x, sel, rw = _moe_inputs(case, seed)
    T, E, H, I, topk = case["tokens"], case["experts"], case["hidden"], case["inter"], case["topk"]
    table = lambda i, j: torch.tensor([e[i][j].data_ptr() for e in experts], dtype=torch.long, device=DEV)
    state = {"kind": "moe", "keep": experts, "tables": [table(i, j) for i in range(3) for j in range(3)], "x": x,
             "bits": torch.tensor(_expert_K(case), dtype=torch.uint8, device=DEV),
             "out": torch.zeros((T, H), dtype=torch.float, device=DEV)}
    z = lambda *shape, dt=torch.half: torch.zeros(shape, dtype=dt, device=DEV)
    if T <= 16:                                    # decode: the fused cooperative call and its scratch
        slots = T * topk
        state.update(sel=sel, rw=rw, hidden=H,
                     scratch=[z(slots, H), z(slots, H), z(slots, I, dt=torch.float), z(slots, I, dt=torch.float),
                              z(slots, I), z(slots, H, dt=torch.float),
                              torch.zeros(ops.moe_coop_ctr_len(slots, T, I, H), dtype=torch.int32, device=DEV)])
        return state
    flat = sel.reshape(-1)                         # prompt: assignments sorted by expert, pooled buffers
    order = torch.argsort(flat, stable=True)
    count = torch.bincount(flat, minlength=E + 1)
    conc = ops.exl3_moe_max_concurrency(torch.cuda.current_device())
    pool = -(-T * topk // conc)
    state.update(count=count, tokens=order // topk, weights=rw.reshape(-1)[order].contiguous(),
                 active=int((count[:E] > 0).sum()),
                 scratch=[z(conc, pool, H), z(conc, pool, H), z(conc, pool, I), z(conc, pool, I)])
    return state


# ------------------------------------------------------------------ one pass
def run(state):
    kind = state["kind"]
    if kind == "linear":
        return state["layer"](state["x"])
    if kind == "qkv":
        return state["bundle"].run(state["x"])
    if kind == "step":
        stack = state["stack"]
        out = stack(state["x"])
        # the normed row, the residual stream, and of what goes to the cache each layer's v row
        return [out, stack.h] + [qkv.outs[2] for qkv in stack.qkv]
    out, tabs, bits = state["out"], state["tables"], state["bits"]
    if "sel" in state:
        ops.exl3_moe_coop(state["x"], state["sel"], state["rw"], -1, -1, state["hidden"], *tabs, None, None, None,
                          4.0, 4.0, 4.0, False, True, ops.MOE_ACT["silu"], 0.0, True, *state["scratch"], out,
                          None, None, bits, bits, bits)
        return out
    out.zero_()                                    # exl3_moe adds into its output
    ops.exl3_moe(state["x"], out, state["count"], state["tokens"], state["weights"], *state["scratch"],
                 ops.MOE_ACT["silu"], 0.0, 0.0, 0.0, *tabs, False, True, False, True, False, True, 0.0, state["active"],
                 bits_g=bits, bits_u=bits, bits_d=bits)
    return out


# ------------------------------------------------------------------ what a pass cannot do without
def _linear_work(rows, k, n, K):
    return k * n * K / 8 + 2 * (rows * (k + n) + k + n), 2.0 * rows * k * n


def work(case):
    kind = case["kind"]
    if kind == "linear":
        b, f = _linear_work(case["rows"], case["k"], case["n"], case["K"])
    elif kind == "qkv":
        b, f = _linear_work(case["rows"], case["k"], case["n"] + 2 * case["kv"], case["K"])
    elif kind == "step":
        H, V, I = case["hidden"], case["kv"], case["inter"]
        weights = H * (H + 2 * V) + H * H + 2 * H * I + I * H
        b, f = case["layers"] * (weights * case["K"] / 8 + 4 * V), case["layers"] * 2.0 * weights
    else:
        E, T, topk = case["experts"], case["tokens"], case["topk"]
        weights = 3 * case["hidden"] * case["inter"]
        touched = E * (1 - (1 - topk / E) ** T)    # experts that T tokens reach, on average
        mean_K = sum(_expert_K(case)) / E
        b, f = touched * weights * mean_K / 8 + T * case["hidden"] * 6, 2.0 * T * topk * weights
    return {"bytes": b, "flops": f}


def tolerance(case):
    """fp16 inputs and outputs around fp32 sums: a linear rounds the rotated input and the result
    (measured 3.7e-4 to 4.9e-4 from float64), from 2048 rows the unrotated weight instead (9.5e-4);
    a routed expert also rounds its activation (5.1e-4 in fp32 scratch, 9.1e-4 in fp16); a step
    carries every layer's roundings to its end (3.4e-3 at 32 layers).  About four times what was
    measured."""
    if case["kind"] == "step":
        return {"rel": 0.014}
    if case["kind"] == "linear" and case["rows"] >= 2048 or case["kind"] == "moe" and case["tokens"] > 16:
        return {"rel": 4e-3}
    return {"rel": 2e-3}


# ------------------------------------------------------------------ float64
_MUL = {"3inst": (89226354, 64248484), "mcg": (0xCBAC1FED, 0), "mul1": (0x83DCD12D, 0)}


def _weights64(trellis, K, cb):
    """The float64 values of a trellis' fp16 weights (k, n), rotated basis."""
    kt, nt, width = trellis.shape
    words = trellis.to(torch.int64) & 0xFFFF
    words = words.view(kt, nt, width // 2, 2).flip(-1).reshape(kt, nt, width)      # most significant bit first
    pos = torch.arange(256, device=DEV)
    b = int(K)
    end = (pos + 1) * b if K == b else (pos >> 1) * (2 * b + 1) + torch.where(pos % 2 == 1, 2 * b + 1, b)
    start = (end - 16) % (16 * width)
    i, off = start // 16, start % 16
    state = (((words[..., i] << 16) | words[..., (i + 1) % width]) >> (16 - off)) & 0xFFFF
    mul, add = _MUL[cb]
    x = (state * mul + add) & 0xFFFFFFFF
    if cb == "mul1":
        total = (x & 255) + ((x >> 8) & 255) + ((x >> 16) & 255) + (x >> 24)
        scale, shift = (torch.tensor([v], dtype=torch.int16).view(torch.half).item() for v in (0x1EEE, 0xC931 - 65536))
        val = ((1024 + total).float() * scale + shift).half()                      # exact in fp32, rounded once
    else:
        x = (x & 0x8FFF8FFF) ^ 0x3B603B60
        as_half = lambda v: torch.where(v >= 32768, v - 65536, v).to(torch.int16).view(torch.half)
        val = as_half(x & 0xFFFF) + as_half(x >> 16)
    lane, j = pos // 8, pos % 8                    # where a tile's positions lie in its 16 x 16 block
    row = (lane % 4) * 2 + torch.tensor([0, 1, 8, 9], device=DEV)[j % 4]
    col = lane // 4 + torch.where(j >= 4, 8, 0)
    tile = torch.empty(kt, nt, 256, dtype=torch.half, device=DEV)
    tile[..., row * 16 + col] = val
    return tile.view(kt, nt, 16, 16).permute(0, 2, 1, 3).reshape(kt * 16, nt * 16).double()


def _had(x):
    h = torch.ones(1, 1, dtype=torch.float64, device=DEV)
    for _ in range(7):
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
    return (x.reshape(-1, 128) @ (h / math.sqrt(128.0))).view(x.shape)


def _linear64(x, m, K, cb, columns=16384):
    t, suh, svh = m
    xr = _had(x * suh.double())
    parts = [xr @ _weights64(t[:, c:c + columns // 16], K, cb) for c in range(0, t.size(1), columns // 16)]
    return _had(torch.cat(parts, 1)) * svh.double()


def _norm64(h, w):
    return h / torch.sqrt((h * h).mean(-1, keepdim=True) + 1e-5) * w.double()


def exact(case, seed):
    if case["kind"] == "linear":
        m, bias, x = _linear_inputs(case, seed)
        y = _linear64(x.double(), m, case["K"], case["cb"])
        return y if bias is None else y + bias.double()
    if case["kind"] == "qkv":
        mats, x = _qkv_inputs(case, seed)
        return [_linear64(x[0].double(), m, case["K"], case["cb"])[None] for m in mats]
    if case["kind"] == "step":
        layers, final, x = _step_inputs(case, seed)
        lin = lambda v, m: _linear64(v, m, case["K"], case["cb"])
        h, cache = x.double(), []
        for mats, a, b in layers:
            r = _norm64(h, a)
            cache.append(lin(r, mats["v"])[None])
            h = h + lin(lin(r, mats["q"]), mats["o"])
            r = _norm64(h, b)
            h = h + lin(torch.nn.functional.silu(lin(r, mats["gate"])) * lin(r, mats["up"]), mats["down"])
        return [_norm64(h, final), h] + cache
    experts, x, sel, rw = _moe_inputs(case, seed)
    out = torch.zeros(case["tokens"], case["hidden"], dtype=torch.float64, device=DEV)
    for e, K in enumerate(_expert_K(case)):
        tok, slot = (sel == e).nonzero(as_tuple=True)
        if tok.numel() == 0:
            continue
        xe = x[tok].double()
        g, u = (_linear64(xe, experts[e][i], K, "mul1") for i in (0, 1))
        y = _linear64(torch.nn.functional.silu(g) * u, experts[e][2], K, "mul1")
        out.index_add_(0, tok, y * rw[tok, slot].double()[:, None])
    return out
