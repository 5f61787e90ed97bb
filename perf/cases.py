"""The work a serving engine has this framework do, as cases to be timed.

One pass is what one engine step asks of one transformer layer: the bound plan
operations of lunaflux_amd.fp8 / lunaflux_amd.moe, launched on the runtime's
stream and left in flight, as the step executor launches them. Weights and
activations are synthetic (N(0, 0.02) weights quantized to e4m3, N(0, 1) bf16
activations), drawn from the seed.

Two kinds of case:

  layer  the projections of one decoder layer: qkv, o and the gated MLP.
         Widths are Llama-3-8B's (hidden 4096, intermediate 14336, 4096 query
         and 1024 key and value columns), whole or as one rank's share of a
         tensor-parallel group, or a small model's.
  moe    one routed expert MLP, from router logits to the combined rows

`profile` is the launch profile the operations are bound for (its largest row
count); `rows` / `tokens` are live in the step.
"""
import ctypes
import math

import numpy as np
import torch

from lunaflux_amd import fp8, moe

NORM_EPSILON = 1e-5

# Widths of one layer: hidden, query columns, key (= value) columns, intermediate.
LLAMA = dict(hidden=4096, nq=4096, nkv=1024, inter=14336)  # Llama-3-8B
SMALL = dict(hidden=512, nq=512, nkv=512, inter=1536)


def _shard(tp):
    """One rank's share of the Llama layer in a tensor-parallel group of `tp`."""
    return dict(hidden=4096, nq=4096 // tp, nkv=1024 // tp, inter=14336 // tp)


# name: (experts, top_k, hidden, expert intermediate, scale group, route mode)
MOE_MODELS = {
    "mixtral": (8, 2, 4096, 14336, 0, moe.ROUTE_TOPK_SOFTMAX),
    "fine": (64, 6, 2048, 1408, 128, moe.ROUTE_SOFTMAX_TOPK),
}


def listed():
    return [
        # A small (draft) model's layer for a few tokens: launch latency.
        dict(name="small_m4", kind="layer", family="w8a16", scale="channel", **SMALL, rows=4, profile=16, norm=False),
        # One user generating: every weight is read for a single row.
        dict(name="decode_m1", kind="layer", family="w8a16", scale="channel", **LLAMA, rows=1, profile=16, norm=False),
        # Ordinary continuous-batching decode.
        dict(name="decode_m32", kind="layer", family="w8a16", scale="channel", **LLAMA, rows=32, profile=32, norm=False),
        # A larger, ragged batch on one of two tensor-parallel ranks.
        dict(name="decode_tp2_m61", kind="layer", family="w8a16", scale="channel", **_shard(2), rows=61, profile=64,
             norm=False),
        # The largest decode batch of the bf16-activation family.
        dict(name="decode_m128", kind="layer", family="w8a16", scale="channel", **LLAMA, rows=128, profile=128, norm=False),
        # Decode of a checkpoint with 128 x 128 block scales.
        dict(name="decode_block_m24", kind="layer", family="w8a16", scale="block", **LLAMA, rows=24, profile=32, norm=False),
        # One ragged chunk of a chunked prefill.
        dict(name="prefill_m509", kind="layer", family="w8a8", scale="channel", **LLAMA, rows=509, profile=512, norm=False),
        # A long prompt, or many prompts at once; the norm fused with the quantizer.
        dict(name="prefill_m8192", kind="layer", family="w8a8", scale="channel", **LLAMA, rows=8192, profile=8192,
             norm=True),
        # Prefill of a block-scaled checkpoint.
        dict(name="prefill_block_m2048", kind="layer", family="w8a8", scale="block", **LLAMA, rows=2048, profile=2048,
             norm=False),
        # Expert MLP of a few large experts with a skewed load.
        dict(name="mixtral_t1024", kind="moe", model="mixtral", tokens=1024, profile=1024),
        # Many small experts: decode (most see a few rows) and prefill.
        dict(name="fine_moe_t32", kind="moe", model="fine", tokens=32, profile=32),
        dict(name="fine_moe_t4096", kind="moe", model="fine", tokens=4096, profile=4096),
    ]


def _log_uniform(rng, low, high):
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high + 1))) - 0.5))))


def _profile(rows):
    """The smallest launch profile of the usual power-of-two ladder that holds `rows`."""
    return max(16, 1 << (rows - 1).bit_length())


def draw(rng):
    taken = [{k: v for k, v in c.items() if k != "name"} for c in listed()]
    while True:
        case = _draw(rng)
        if case not in taken:
            return case


def _draw(rng):
    kind = rng.choice(["small", "decode", "decode", "decode", "prefill", "prefill", "prefill", "moe", "moe"])
    if kind == "small":
        widths = {name: 128 * rng.randint(2, 12) for name in ("hidden", "nq", "nkv", "inter")}
        rows = _log_uniform(rng, 1, 32)
        return dict(kind="layer", family="w8a16", scale="channel", **widths, rows=rows, profile=_profile(rows), norm=False)
    if kind == "decode":
        rows = _log_uniform(rng, 1, 128)
        return dict(kind="layer", family="w8a16", scale=rng.choice(["channel", "channel", "block"]),
                    **_shard(rng.choice([1, 1, 2, 4])), rows=rows, profile=_profile(rows), norm=False)
    if kind == "prefill":
        scale = rng.choice(["channel", "channel", "block"])
        rows = _log_uniform(rng, 129, 8192 if scale == "channel" else 4096)
        return dict(kind="layer", family="w8a8", scale=scale, **_shard(rng.choice([1, 1, 2])), rows=rows,
                    profile=_profile(rows), norm=scale == "channel" and rng.random() < 0.5)
    model = rng.choice(["mixtral", "fine", "fine"])
    tokens = _log_uniform(rng, 8, 1024 if model == "mixtral" else 4096)
    return dict(kind="moe", model=model, tokens=tokens, profile=_profile(tokens))


# -- inputs, from the seed ----------------------------------------------------

def _quantize_weight(w, block):
    """e4m3 codes (as float8) and fp32 scales of fp32 weights [N, K]: absmax
    over a row, or over a 128 x 128 block."""
    n, k = w.shape
    g = w.view(n // 128, 128, k // 128, 128) if block else w.view(n, 1, 1, k)
    amax = g.abs().amax(dim=(1, 3), keepdim=True)
    q = (g * (448.0 / amax)).to(torch.float8_e4m3fn).view(n, k)
    scales = (amax / 448.0).view(n // 128, k // 128) if block else (amax / 448.0).view(n)
    return q, scales


class _Draws:
    """The seeded draws of one case, in a fixed order."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(seed)

    def normal(self, *shape):
        return torch.randn(*shape, generator=self.g, device="cuda")

    def activations(self, rows, columns):
        return self.normal(rows, columns).to(torch.bfloat16)

    def weight(self, n, k, block):
        return _quantize_weight(self.normal(n, k) * 0.02, block)

    def expert_weights(self, experts, n, k, block):
        parts = [self.weight(n, k, block) for _ in range(experts)]
        return torch.stack([q.view(torch.uint8) for q, _ in parts]).view(torch.float8_e4m3fn), \
            torch.stack([s for _, s in parts])


def _router_logits(draws, model, tokens, experts):
    """N(0, 1) logits plus a popularity bias per expert: N(0, 1.5) (mixtral) or
    Zipf(1.1) by a random ranking (fine)."""
    logits = draws.normal(tokens, experts)
    if model == "mixtral":
        return logits + 1.5 * draws.normal(experts)
    ranks = torch.randperm(experts, generator=draws.g, device="cuda") + 1
    return logits - 1.1 * torch.log(ranks.float())


def _inputs(case, seed):
    """Every input of a case as torch tensors on the GPU; weights as (codes, scales)."""
    d = _Draws(seed)
    if case["kind"] == "layer":
        hidden, nq, nkv, inter = (case[name] for name in ("hidden", "nq", "nkv", "inter"))
        block, m = case["scale"] == "block", case["rows"]
        t = dict(x=d.activations(m, hidden), a=d.activations(m, nq), m=d.activations(m, hidden))
        if case["norm"]:
            t["gamma"] = (1.0 + 0.1 * d.normal(hidden)).to(torch.bfloat16)
            t["win"] = d.weight(nq + 2 * nkv, hidden, block)
        else:
            t["wq"], t["wk"], t["wv"] = (d.weight(n, hidden, block) for n in (nq, nkv, nkv))
        t["wo"] = d.weight(hidden, nq, block)
        t["wg"], t["wu"] = d.weight(inter, hidden, block), d.weight(inter, hidden, block)
        t["wd"] = d.weight(hidden, inter, block)
        return t
    experts, _, hidden, inter, group, _ = MOE_MODELS[case["model"]]
    return dict(x=d.activations(case["tokens"], hidden),
                logits=_router_logits(d, case["model"], case["tokens"], experts),
                wg=d.expert_weights(experts, inter, hidden, group == 128),
                wu=d.expert_weights(experts, inter, hidden, group == 128),
                wd=d.expert_weights(experts, hidden, inter, group == 128))


# -- the framework's side -----------------------------------------------------

_runtime = None


def _rt():
    """The process's runtime: one context, stream and loaded code object."""
    global _runtime
    if _runtime is None:
        torch.cuda.init()
        _runtime = fp8.ProjectionRuntime(0)
    return _runtime


class _Rows:
    """A device allocation's first rows as an array torch can wrap (it keeps
    the allocation). Device addresses do not cross the framework's boundary,
    so the address is taken from the allocation's handle: {vtable, magic and
    kind, counters, flag, parent, base, size}."""

    def __init__(self, allocation, shape):
        self.allocation = allocation
        words = (ctypes.c_uint64 * 8).from_address(allocation.ptr)
        if words[1] & 0xFFFFFFFF != 0x4C464855 or words[7] != allocation.byte_count:
            raise RuntimeError("unexpected allocation handle")
        self.__cuda_array_interface__ = dict(shape=shape, typestr="<i2", data=(int(words[6]), False),
                                             strides=None, version=2)


def _view(allocation, rows, columns):
    return torch.as_tensor(_Rows(allocation, (rows, columns)), device="cuda").view(torch.bfloat16)


def _region(allocation):
    return allocation.region(0, allocation.byte_count, 256)


def _activation(rt, x, profile):
    """The profile-sized activation region holding the live rows of x."""
    a = rt.context.allocate(profile * x.shape[1] * x.element_size())
    a.copy_from_host(x.view(torch.uint8).cpu().numpy())
    return a


def _upload_weight(rt, weight, block):
    q, s = weight
    return rt.upload_weight(q.view(torch.uint8).cpu().numpy(), s.cpu().numpy(),
                            fp8.BLOCK128 if block else fp8.PER_CHANNEL)


class _State:
    """Bound operations, their output views and what they read."""

    def __init__(self):
        self.operations, self.outputs, self.keep = [], [], []


def prepare(case, seed):
    rt = _rt()
    t = _inputs(case, seed)
    s = _State()
    if case["kind"] == "moe":
        _prepare_moe(rt, case, t, s)
    else:
        _prepare_layer(rt, case, t, s)
    return s


def _prepare_layer(rt, case, t, s):
    m, profile, family, block = case["rows"], case["profile"], case["family"], case["scale"] == "block"
    hidden, packed = case["hidden"], case["nq"] + 2 * case["nkv"]
    counts = rt.step_counts(m, decode=family == "w8a16")
    w = {name: _upload_weight(rt, v, block) for name, v in t.items() if isinstance(v, tuple)}
    x = {name: _activation(rt, t[name], profile) for name in ("x", "a", "m")}

    def output(columns):
        y = rt.context.allocate(profile * columns * 2)
        s.outputs.append(_view(y, m, columns))
        return _region(y)

    if case["norm"]:
        gamma = rt.context.upload(t["gamma"].view(torch.int16).cpu().numpy())
        xq = rt.context.allocate(fp8.act_quant_bytes(profile, hidden))
        s.operations.append(fp8.BoundOperation([
            rt.bind_rms_norm_quant(counts, _region(x["x"]), _region(gamma), w["win"], _region(xq), profile,
                                   NORM_EPSILON),
            rt.bind_dense_quantized(counts, _region(xq), w["win"], output(packed), profile)]))
        s.keep += [gamma, xq]
    else:
        s.operations.append(rt.bind_qkv(family, counts, _region(x["x"]), w["wq"], w["wk"], w["wv"],
                                        output(packed), profile))
    s.operations.append(rt.bind_dense(family, counts, _region(x["a"]), w["wo"], output(hidden), profile))
    s.operations.append(rt.bind_gated_mlp(family, counts, _region(x["m"]), w["wg"], w["wu"], w["wd"],
                                          output(hidden), profile))
    s.keep += [counts, w, x]


def _prepare_moe(rt, case, t, s):
    experts, top_k, hidden, inter, group, mode = MOE_MODELS[case["model"]]
    tokens, profile = case["tokens"], case["profile"]
    desc = moe.moe_descriptor(experts, top_k, mode, hidden, inter, group)
    desc_region = rt.context.upload(desc.as_bytes())
    counts = rt.step_counts(tokens, decode=False)
    x, logits = _activation(rt, t["x"], profile), _activation(rt, t["logits"], profile)
    w = [_upload_weight(rt, t[name], group == 128) for name in ("wg", "wu", "wd")]
    out = rt.context.allocate(profile * hidden * 2)
    s.outputs.append(_view(out, tokens, hidden))
    s.operations.append(moe.bind_moe(rt, counts, desc, desc_region.region(0, 32, 4), _region(logits), _region(x),
                                     *w, _region(out), profile))
    s.keep += [desc_region, counts, x, logits, w]


def run(state):
    stream = _rt().stream
    for operation in state.operations:
        operation.launch(stream, synchronous=False)
    return list(state.outputs)


# -- work, tolerance and the 64-bit result ------------------------------------

def _touched_experts(model, tokens):
    """Expected number of experts with rows, over a few draws of the router."""
    experts, top_k = MOE_MODELS[model][:2]
    rng, total = np.random.default_rng(5), 0
    for _ in range(8):
        logits = rng.standard_normal((tokens, experts))
        logits += 1.5 * rng.standard_normal(experts) if model == "mixtral" else -1.1 * np.log(np.arange(1, experts + 1))
        total += np.unique(np.argpartition(-logits, top_k - 1, axis=1)[:, :top_k]).size
    return total / 8


def work(case):
    def dense(m, k, n, block=False):
        return n * k + 4 * (n * k // 16384 if block else n) + 2 * m * (k + n), 2 * m * n * k

    if case["kind"] == "layer":
        m, block = case["rows"], case["scale"] == "block"
        hidden, nq, nkv, inter = (case[name] for name in ("hidden", "nq", "nkv", "inter"))
        parts = [dense(m, hidden, nq + 2 * nkv, block), dense(m, nq, hidden, block),
                 dense(m, hidden, 2 * inter, block), dense(m, inter, hidden, block)]
        parts.append((-2 * m * (2 * inter + inter), 0))  # gate, up and h stay inside the MLP
    else:
        experts, top_k, hidden, inter, _, _ = MOE_MODELS[case["model"]]
        t = case["tokens"]
        parts = [(3 * hidden * inter * _touched_experts(case["model"], t) + 4 * t * hidden + 4 * t * experts,
                  6 * t * top_k * hidden * inter)]
    return {"bytes": float(sum(b for b, _ in parts)), "flops": float(sum(f for _, f in parts))}


def tolerance(case):
    # About four times the distance from the 64-bit result: 1.7e-3 from the bf16
    # outputs' own rounding; 2.1e-3 to 2.9e-3 where a hidden row is quantized to
    # e4m3 on the way (its rounding moves a few codes) or bf16 rows are combined.
    return {"rel": 7e-3 if case.get("family") == "w8a16" else 1.1e-2}


def _dequantized(weight, block):
    q, s = weight
    q = q.double()
    if not block:
        return q * s.double()[:, None]
    return q * s.double().repeat_interleave(128, 0).repeat_interleave(128, 1)


def _quantized(x, group=None):
    """The activation quantizer of the W8A8 family, dequantized: per row, or per
    128 columns of a row."""
    rows, columns = x.shape
    g = x.float().view(rows, -1, group or columns)
    amax = g.abs().amax(dim=2, keepdim=True)
    # (through 64 bits: torch divides a scalar by a tensor with a reciprocal)
    ratio, scale = (448.0 / amax.double()).float(), (amax.double() / 448.0).float()
    q = (g * ratio).to(torch.float8_e4m3fn).double()
    return torch.where(amax > 0, q * scale.double(), 0.0).view(rows, columns)


def _silu_gated(g, u):
    return g / (1.0 + torch.exp(-g)) * u


def exact(case, seed):
    """run()'s result with every product and sum in 64 bits. What the path
    defines is kept: e4m3 activations in the W8A8 family and the experts, and a
    bf16 hidden row between the halves of an MLP."""
    t = _inputs(case, seed)
    if case["kind"] == "moe":
        return [_exact_moe(case, t).cpu()]
    block = case["scale"] == "block"

    def activation(x):
        if case["family"] == "w8a16":
            return x.double()
        return _quantized(x, 128 if block else None)

    def dense(x, *weights):
        return torch.cat([activation(x) @ _dequantized(w, block).t() for w in weights], dim=1)

    if case["norm"]:
        x = t["x"].double()
        normed = x / torch.sqrt(x.square().mean(dim=1, keepdim=True) + NORM_EPSILON) * t["gamma"].double()
        outputs = [dense(normed, t["win"])]
    else:
        outputs = [dense(t["x"], t["wq"], t["wk"], t["wv"])]
    outputs.append(dense(t["a"], t["wo"]))
    hidden = _silu_gated(dense(t["m"], t["wg"]), dense(t["m"], t["wu"])).to(torch.bfloat16)
    outputs.append(dense(hidden, t["wd"]))
    return [y.cpu() for y in outputs]


def _exact_moe(case, t):
    experts, top_k, hidden, _, group, mode = MOE_MODELS[case["model"]]
    logits = t["logits"].double()
    top, ids = torch.topk(logits, top_k, dim=1)
    weights = torch.softmax(top, 1) if mode == moe.ROUTE_TOPK_SOFTMAX else torch.softmax(logits, 1).gather(1, ids)
    x = _quantized(t["x"], group or None)
    out = torch.zeros(case["tokens"], hidden, dtype=torch.float64, device="cuda")
    for e in range(experts):
        rows, slot = (ids == e).nonzero(as_tuple=True)
        if rows.numel() == 0:
            continue
        wg, wu, wd = (_dequantized((t[n][0][e], t[n][1][e]), group == 128) for n in ("wg", "wu", "wd"))
        xe = x[rows]
        h = _silu_gated(xe @ wg.t(), xe @ wu.t()).to(torch.bfloat16)
        y = _quantized(h, group or None) @ wd.t()
        out.index_add_(0, rows, y * weights[rows, slot][:, None])
    return out
