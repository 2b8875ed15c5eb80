"""The work that a user of this framework has it do, as cases that can be timed and checked.

A serving program meets the framework in four places, and each has a kind of case here:

* ``linear``: one ``exactmm::linear`` call on packed weights, launched eagerly, as prefill and
  every step outside a captured graph run it. Any row count from one token to a long prompt,
  shapes the tuning tables list and shapes they do not, bf16 and fp16 rows, F = 14 and F = 15.
* ``step``: the four linears (qkv, o, gate_up, down) of some layers at a decode batch, captured
  once in a graph and replayed for every token, as a decode step runs them.
* ``attention``: the paged decode attention of some layers, captured the same way (or launched
  eagerly with the count of decode requests on the GPU, as in a step that also prefills).
* ``load``: digitizing and packing one weight matrix when a model is loaded.

The exact linears promise the same bits for every schedule, so their tolerance is "exact".
"""
import sys
from pathlib import Path

import torch

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "vllm-exact_amd"))

import vllm_exact  # noqa: E402
from vllm_exact import paged_attn, plugin  # noqa: E402

LAYER = {"qkv": (6144, 4096), "o": (4096, 4096), "gate_up": (24576, 4096), "down": (4096, 12288)}
# (N, K) pairs the shipped tuning tables hold, and the largest linear pass that is drawn.
TABLED = ((6144, 4096), (4096, 4096), (24576, 4096), (4096, 12288), (10240, 4096), (12288, 4096), (64, 4096))
MOST_PRODUCTS = 4096 * 24576 * 4096
MOST_KV = 64 * 8192 * 8 * 128


def listed():
    return [
        # The smallest call: one token through one square projection, launched eagerly.
        {"name": "linear-1-row", "kind": "linear", "m": 1, "n": 4096, "k": 4096, "dtype": "bf16", "f": 14},
        # A decode step's linears for a single stream: latency and launches.
        {"name": "step-1", "kind": "step", "m": 1, "layers": 4, "f": 14},
        # A small batch at the 15-bit setting (four dots).
        {"name": "step-16-f15", "kind": "step", "m": 16, "layers": 4, "f": 15},
        # Ordinary and large decode batches.
        {"name": "step-64", "kind": "step", "m": 64, "layers": 3, "f": 14},
        {"name": "step-256", "kind": "step", "m": 256, "layers": 3, "f": 14},
        # The exact lm_head over a batch's last tokens.
        {"name": "lm-head-256", "kind": "linear", "m": 256, "n": 151936, "k": 4096, "dtype": "bf16", "f": 14},
        # A long prompt through the widest linear of a layer: the largest work.
        {"name": "prefill-4096", "kind": "linear", "m": 4096, "n": 24576, "k": 4096, "dtype": "bf16", "f": 14},
        # A ragged prompt in fp16 through a layer of another model, which the tables do not list.
        {"name": "prefill-1531-fp16", "kind": "linear", "m": 1531, "n": 5136, "k": 2600, "dtype": "fp16", "f": 14},
        # One long request, decoded alone.
        {"name": "attention-1x16k", "kind": "attention", "batch": 1, "context": 16384, "heads": 32, "kv_heads": 8,
         "dim": 128, "page": 16, "max_len": 16384, "layers": 8, "ragged": False, "mixed": False},
        # A loaded server: 64 requests of up to 8K tokens, lengths spread.
        {"name": "attention-64x8k", "kind": "attention", "batch": 64, "context": 8192, "heads": 32, "kv_heads": 8,
         "dim": 128, "page": 16, "max_len": 16384, "layers": 2, "ragged": True, "mixed": False},
        # A step that also prefills: wide heads on large pages, the decode count on the GPU.
        {"name": "attention-12x3k-mixed", "kind": "attention", "batch": 12, "context": 3000, "heads": 16,
         "kv_heads": 2, "dim": 256, "page": 528, "max_len": 16384, "layers": 4, "ragged": True, "mixed": True},
        # Loading a model: one wide weight matrix.
        {"name": "load-24576x4096", "kind": "load", "n": 24576, "k": 4096, "dtype": "bf16", "f": 14},
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(("linear", "linear", "step", "attention", "attention", "load"))
    f = 15 if rng.random() < 0.25 else 14
    if kind == "step":
        m = _log_int(rng, 1, 512)
        return {"kind": kind, "m": m, "layers": rng.randint(2, 4), "f": f}
    if kind == "attention":
        heads, kv_heads = rng.choice(((32, 8), (16, 2), (32, 4), (16, 8), (8, 8)))
        dim = rng.choice((64, 128, 128, 256))
        context = _log_int(rng, 64, 16384)
        most = max(1, MOST_KV // (context * kv_heads * dim))
        return {"kind": kind, "batch": min(256, _log_int(rng, 1, most)), "context": context, "heads": heads,
                "kv_heads": kv_heads, "dim": dim, "page": rng.choice((16, 16, 32, 64, 528)), "max_len": 16384,
                "layers": rng.randint(1, 2) if context > 4096 else rng.randint(2, 8),
                "ragged": rng.random() < 0.7, "mixed": rng.random() < 0.25}
    if rng.random() < 0.5:
        n, k = rng.choice(TABLED)
    else:
        n, k = _log_int(rng, 512, 16384), _log_int(rng, 512, 12288)
        if rng.random() < 0.6:  # most models' sizes are round
            n, k = -(-n // 256) * 256, -(-k // 256) * 256
    dtype = "fp16" if rng.random() < 0.25 else "bf16"
    if kind == "load":
        return {"kind": kind, "n": n, "k": k, "dtype": dtype, "f": f}
    return {"kind": kind, "m": _log_int(rng, 1, min(16384, MOST_PRODUCTS // (n * k))), "n": n, "k": k,
            "dtype": dtype, "f": f}


# ---------------------------------------------------------------------------------- inputs
def _dtype(case):
    return torch.float16 if case.get("dtype") == "fp16" else torch.bfloat16


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _activations(g, m, k, dtype):
    """N(0, 1) rows of mixed magnitude with a few outlier channels, as hidden states have them."""
    x = torch.randn(m, k, device="cuda", generator=g)
    x *= 10 ** (torch.rand(m, 1, device="cuda", generator=g) * 2 - 1)
    x[:, torch.randint(0, k, (4,), device="cuda", generator=g)] *= 20
    return x.to(dtype)


def _weights(g, n, k, dtype):
    """N(0, 0.02), in row blocks so that the fp32 temporaries stay small."""
    w = torch.empty(n, k, device="cuda", dtype=dtype)
    for i in range(0, n, 32768):
        w[i:i + 32768] = torch.randn(min(32768, n - i), k, device="cuda", generator=g) * 0.02
    return w


def _settings(f):
    """What enable() sets for a program that asks for F = f."""
    plugin.F = f
    plugin.TRUNC = f == 14
    plugin.load_table((vllm_exact.TABLES_F15 if f == 15 else vllm_exact.TABLES)["mi355x"])


def _linear_inputs(case, seed):
    """x and the bf16/fp16 weights of a linear or step case: a list of (x, w)."""
    g = _generator(seed)
    if case["kind"] == "linear":
        return [(_activations(g, case["m"], case["k"], _dtype(case)), _weights(g, case["n"], case["k"], _dtype(case)))]
    return [(_activations(g, case["m"], k, torch.bfloat16), _weights(g, n, k, torch.bfloat16))
            for _ in range(case["layers"]) for n, k in LAYER.values()]


def _attention_inputs(case, seed):
    """Queries, caches in vLLM's FlashAttention layout [blocks, KV, page, 2 D], block tables
    over permuted pages, lengths in [context / 2, context], and the decode count."""
    g = _generator(seed)
    b, page, d, kv = case["batch"], case["page"], case["dim"], case["kv_heads"]
    pages = -(-case["context"] // page)
    blocks = b * pages + 3
    state = {"q": [], "kv": [], "bt": [], "out": []}
    for _ in range(case["layers"]):
        state["q"].append(torch.randn(b, case["heads"], d, device="cuda", generator=g).to(torch.bfloat16))
        state["kv"].append(torch.empty(blocks, kv, page, 2 * d, device="cuda", dtype=torch.bfloat16).normal_(generator=g))
        state["out"].append(torch.zeros(b, case["heads"], d, device="cuda", dtype=torch.bfloat16))
        state["bt"].append(torch.randperm(blocks, device="cuda", generator=g)[:b * pages].view(b, pages).to(torch.int32))
    lo = max(1, case["context"] // 2) if case["ragged"] else case["context"]
    state["sl"] = torch.randint(lo, case["context"] + 1, (b,), device="cuda", generator=g).to(torch.int32)
    state["live"] = torch.tensor([max(1, 3 * b // 4)], device="cuda", dtype=torch.int32) if case["mixed"] else None
    return state


# ---------------------------------------------------------------------------------- passes
def _linears(state):
    return [torch.ops.exactmm.linear(x, *w) for x, w in state["pairs"]]


def _attend(state):
    case = state["case"]
    for q, kv, bt, out in zip(state["q"], state["kv"], state["bt"], state["out"]):
        key, value = kv.transpose(1, 2).split(case["dim"], dim=-1)
        paged_attn.paged_decode(q, key, value, bt, state["sl"], case["dim"] ** -0.5, out, case["batch"],
                                case["context"], n_live=state["live"])
    return state["out"]


def _capture(call, state):
    """The step in a graph, after one eager pass on a side stream as torch asks for."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        call(state)
    torch.cuda.current_stream().wait_stream(side)
    state["graph"] = torch.cuda.CUDAGraph()
    with torch.cuda.graph(state["graph"]):
        state["result"] = call(state)
    return state


def prepare(case, seed):
    if case["kind"] == "attention":
        paged_attn.MAX_LEN = case["max_len"]
        state = _attention_inputs(case, seed)
        state["case"] = case
        return state if case["mixed"] else _capture(_attend, state)
    _settings(case["f"])
    if case["kind"] == "load":
        return {"case": case, "w": _weights(_generator(seed), case["n"], case["k"], _dtype(case))}
    state = {"case": case, "pairs": [(x, plugin.pack_weight(w)) for x, w in _linear_inputs(case, seed)]}
    return _capture(_linears, state) if case["kind"] == "step" else state


def run(state):
    if "graph" in state:
        state["graph"].replay()
        return state["result"]
    kind = state["case"]["kind"]
    if kind == "attention":
        return _attend(state)
    if kind == "load":
        packed, _, cw, sw = plugin.pack_weight(state["w"])
        return [packed, cw, sw]
    return _linears(state)


# ---------------------------------------------------------------------------------- accounting
def _linear_work(m, n, k, f):
    return 2 * n * k + 2 * m * k + 2 * m * n + 8 * n, (3 if f == 14 else 4) * 2 * m * n * k


def work(case):
    if case["kind"] == "attention":
        mean = (case["context"] * 3 / 4) if case["ragged"] else case["context"]
        rows = max(1, 3 * case["batch"] // 4) if case["mixed"] else case["batch"]
        keys = rows * mean * case["layers"]
        return {"bytes": keys * case["kv_heads"] * case["dim"] * 4 + 4 * rows * case["heads"] * case["dim"] * case["layers"],
                "flops": keys * case["heads"] * case["dim"] * 4}
    if case["kind"] == "load":
        return {"bytes": 4 * case["n"] * case["k"] + 8 * case["n"], "flops": 0}
    if case["kind"] == "linear":
        b, fl = _linear_work(case["m"], case["n"], case["k"], case["f"])
    else:
        parts = [_linear_work(case["m"], n, k, case["f"]) for n, k in LAYER.values()]
        b, fl = (case["layers"] * sum(p[i] for p in parts) for i in (0, 1))
    return {"bytes": b, "flops": fl}


def tolerance(case):
    """Bits for the linears and the digits. The attention's outputs are bf16 of fp32 sums: other
    orders of the sums (segments of 256 to 4096 keys, 16 to 64 keys a step, 4 or 8 waves) moved a
    few values by one bf16 step (0.0078 of the value), 1.5e-4 in the 2-norm at most."""
    return {"rel": 6e-4, "max": 0.016} if case["kind"] == "attention" else "exact"


# ---------------------------------------------------------------------------------- 64 bits
def _digits(t, f):
    """q = trunc(t 2^sh) per row and its low digit, in float64, with the shifts."""
    t = t.double()
    top = t.abs().amax(dim=1)
    sh = f - torch.where(top > 0, torch.frexp(top).exponent, 0)
    q = torch.trunc(t * torch.ldexp(torch.ones_like(top), sh)[:, None])
    low = q % 256 - 128 if f == 15 else (q + 128) % 256 - 128
    return q, low, sh


def _exact_linear(x, w, f):
    """The fixed-point product in float64: whole numbers below 2^53, scaled by powers of two."""
    qx, lx, sx = _digits(x, f)
    out = []
    for i in range(0, w.shape[0], 16384):
        qw, lw, sw = _digits(w[i:i + 16384], f)
        tot = qx @ qw.T
        if f == 14:
            tot -= lx @ lw.T
        out.append(torch.ldexp(tot, -(sx[:, None] + sw[None, :])))
    return torch.cat(out, dim=1)


def _exact_attention(case, seed):
    s = _attention_inputs(case, seed)
    rows = int(s["live"]) if case["mixed"] else case["batch"]
    d, kv, group = case["dim"], case["kv_heads"], case["heads"] // case["kv_heads"]
    outs = []
    for q, cache, bt in zip(s["q"], s["kv"], s["bt"]):
        out = torch.zeros(case["batch"], case["heads"], d, device="cuda", dtype=torch.float64)
        for b in range(rows):
            n = int(s["sl"][b])
            rows_b = cache[bt[b].long()].transpose(0, 1).reshape(kv, -1, 2 * d)[:, :n].double()
            key, value = rows_b[..., :d], rows_b[..., d:].contiguous()
            scores = torch.bmm(key, q[b].double().view(kv, group, d).transpose(1, 2).contiguous()) * d ** -0.5
            p = torch.softmax(scores, dim=1).transpose(1, 2).contiguous()
            out[b] = torch.bmm(p, value).reshape(-1, d)
        outs.append(out)
    return outs


def _exact_load(case, seed):
    """The digits in the packed order (16-row by 64-column blocks, h then l), sums and shifts."""
    q, low, sh = _digits(_weights(_generator(seed), case["n"], case["k"], _dtype(case)), case["f"])
    q = q - 128 if case["f"] == 15 else q
    n, k = case["n"], case["k"]
    planes = torch.zeros(2, -(-n // 16) * 16, -(-k // 64) * 64, device="cuda", dtype=torch.int8)
    planes[0, :n, :k] = torch.div(q - low, 256).to(torch.int8)
    planes[1, :n, :k] = low.to(torch.int8)
    packed = planes.view(2, planes.shape[1] // 16, 16, planes.shape[2] // 64, 4, 16).permute(1, 3, 0, 4, 2, 5)
    sums = q.sum(dim=1) if case["f"] == 15 else torch.zeros(n, device="cuda")
    return [packed.reshape(planes.shape[1] // 16, planes.shape[2] // 64, 2, 1024), sums.to(torch.int32), sh.to(torch.int32)]


def exact(case, seed):
    if case["kind"] == "attention":
        return _exact_attention(case, seed)
    if case["kind"] == "load":
        return _exact_load(case, seed)
    return [_exact_linear(x, w, case["f"]) for x, w in _linear_inputs(case, seed)]
