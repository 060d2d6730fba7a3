"""The framework's measured work: the quantised linears, the routed expert
layer and the generate calls built on them, through the package's public
entry points, over the sizes, types and options they are used at.

listed() names the cases, draw(rng) gives further ones of the same ranges.
A case is a dict of plain values with a "kind":

  linear    Weight.mm_dev / mm_exact_dev / mm_rows_dev of one resident weight
            ("dtype" i8, i4 or q4a; "group" for i4 / q4a) on m rows
  moe       MoeBank.forward_dev: one routed layer of "experts" experts
            ("dtype" i8, i4, q4a or f16) on "tokens" tokens
  generate  Rope / Gemma generate (or generate_batch): prefill of "prompt"
            tokens and "new" greedy tokens on a bundle of "layers" layers of
            the family's widths, logits returned

Weights, activations and prompts are seeded: activations N(0, 1) with 1% of
the channels times 20 (the outlier channels that the int8 path selects),
router logits normal, int8 weights uniform bytes with f16 scales, int4
nibbles uniform with f16 group scales.
"""
import math
import os
import shutil
import tempfile

import numpy as np
import torch

import fieldrun_amd as fa
from fieldrun_amd import synth

OUTLIERS = 32  # per-token outlier channels of the int8 path
# generate's families: (heads, kv heads, head width, d, ffn) of Qwen2.5-0.5B,
# Qwen2.5-7B and Gemma-2-2b
FAMILIES = {
    "rope_896": ("rope", 14, 2, 64, 896, 4864),
    "rope_3584": ("rope", 28, 4, 128, 3584, 18944),
    "gemma_2304": ("gemma", 8, 4, 256, 2304, 9216),
}

_ctx = None


def _context():
    """The program's one context (device 0, its own stream)."""
    global _ctx
    if _ctx is None:
        _ctx = fa.Context(0)
    return _ctx


def listed():
    return [
        # a decode step's smallest linear (Qwen2.5-0.5B gate / up): latency and the launch
        {"name": "i8_decode_small", "kind": "linear", "dtype": "i8", "api": "mm", "m": 1, "k": 896, "n": 4864},
        # a decode step's largest linear (Qwen2.5-7B gate|up): the weight stream
        {"name": "i8_decode_wide", "kind": "linear", "dtype": "i8", "api": "mm", "m": 1, "k": 3584, "n": 37888},
        # decode of a ragged batch of sequences, or a very short prompt
        {"name": "i8_decode_batch", "kind": "linear", "dtype": "i8", "api": "mm", "m": 13, "k": 4096, "n": 14336},
        # a short prompt through a small model, one row over a tile
        {"name": "i8_prompt_129", "kind": "linear", "dtype": "i8", "api": "mm", "m": 129, "k": 896, "n": 4864},
        # a long prompt's prefill linear
        {"name": "i8_prefill", "kind": "linear", "dtype": "i8", "api": "mm", "m": 2048, "k": 4096, "n": 14336},
        # int4 decode (Gemma-2-2b gate|up)
        {"name": "i4_decode", "kind": "linear", "dtype": "i4", "group": 32, "api": "mm", "m": 1, "k": 2304,
         "n": 18432},
        # int4 prefill of a middling prompt (Gemma-2-2b gate)
        {"name": "i4_prefill", "kind": "linear", "dtype": "i4", "group": 32, "api": "mm", "m": 300, "k": 2304,
         "n": 9216},
        # affine int4 prefill of a short prompt (Gemma-2-2b down)
        {"name": "q4a_prefill", "kind": "linear", "dtype": "q4a", "group": 64, "api": "exact", "m": 64, "k": 9216,
         "n": 2304},
        # a Qwen3-MoE routed layer at decode
        {"name": "moe_i8_decode", "kind": "moe", "dtype": "i8", "tokens": 1, "experts": 128, "d": 2048, "mi": 768,
         "topk": 8},
        # the same layer with int4 experts over a prompt
        {"name": "moe_i4_prefill", "kind": "moe", "dtype": "i4", "group": 32, "tokens": 512, "experts": 128,
         "d": 2048, "mi": 768, "topk": 8},
        # a long int8 prompt and a short answer at Qwen2.5-7B's widths
        {"name": "rope_i8_generate", "kind": "generate", "family": "rope_3584", "dtype": "int8", "kv_int8": False,
         "layers": 2, "vocab": 16384, "batch": 1, "prompt": 2048, "new": 16},
        # sixteen int4 sequences decoded together at Gemma-2-2b's widths
        {"name": "gemma_i4_batch", "kind": "generate", "family": "gemma_2304", "dtype": "int4", "kv_int8": False,
         "layers": 2, "vocab": 16384, "batch": 16, "prompt": 64, "new": 24},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _rows(rng):
    """Rows of a linear: one token, a decode batch, or a prompt."""
    r = rng.random()
    return 1 if r < 0.3 else rng.randint(2, 16) if r < 0.55 else _log(rng, 17, 2048)


def _width(rng, lo, hi, ragged=0.3):
    """An input width: a multiple of 32 as models have them, or any number."""
    k = _log(rng, lo, hi)
    return k if rng.random() < ragged else max(32, k // 32 * 32)


def draw(rng):
    kind = rng.choice(["i8", "i8", "i4", "i4", "q4a", "moe", "moe", "generate"])
    if kind in ("i8", "i4", "q4a"):
        c = {"kind": "linear", "dtype": kind, "api": "mm", "m": _rows(rng), "k": _width(rng, 256, 16384),
             "n": _log(rng, 64, 40000)}
        if kind != "i8":
            c["group"] = rng.choice([32, 32, 32, 64])
        c["api"] = rng.choice(["mm", "mm", "exact", "rows"] if c["m"] <= 16 and kind == "i4" else ["mm", "mm", "exact"])
        while c["n"] * c["k"] > 3584 * 37888:
            c["n"] //= 2
        most = 2048 * 4096 * 14336 if kind == "i8" else 1024 * 2304 * 9216
        c["m"] = max(1, min(c["m"], most // (c["n"] * c["k"])))
        return c
    if kind == "moe":
        dtype = rng.choice(["i8", "i8", "i4", "i4", "q4a", "f16"])
        e = rng.choice([8, 32, 64, 128]) if dtype in ("i8", "i4") else rng.choice([8, 16])
        c = {"kind": "moe", "dtype": dtype, "tokens": rng.choice([1, _log(rng, 2, 512)]), "experts": e,
             "d": _width(rng, 512, 2048, 0.0), "mi": _width(rng, 256, 1024, 0.0), "topk": rng.randint(1, min(8, e))}
        if dtype in ("i4", "q4a"):
            c["group"] = 32
        return c
    family = rng.choice(sorted(FAMILIES))
    gemma = family.startswith("gemma")
    batch = rng.choice([1, rng.randint(2, 16)])
    return {"kind": "generate", "family": family, "dtype": rng.choice(["int4", "q4a", "int8"] if gemma else
                                                                     ["int8", "int4"]) if family != "rope_3584"
            else "int8", "kv_int8": rng.random() < 0.3, "layers": rng.randint(1, 2),
            "vocab": _log(rng, 1000, 16384), "batch": batch,
            "prompt": _log(rng, 8, 2000 if batch == 1 else 128), "new": _log(rng, 1, 24)}


def _rng(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) & 0x7FFFFFFF)
    return g


def _activations(g, m, k):
    a = torch.randn(m, k, generator=g, device="cuda")
    hot = torch.randperm(k, generator=g, device="cuda")[:max(1, round(0.01 * k))]
    a[:, hot] *= 20.0
    return a


def _f16_uniform(g, lo, hi, *shape):
    return (torch.rand(*shape, generator=g, device="cuda") * (hi - lo) + lo).half()


def _bytes(g, *shape):
    return torch.randint(0, 256, shape, generator=g, device="cuda", dtype=torch.uint8)


def _i8(g, *shape):
    return torch.randint(-127, 128, shape, generator=g, device="cuda", dtype=torch.int8)


def _u16(t):
    """f16 tensor -> host array of its bits."""
    return t.cpu().numpy().view(np.uint16)


def _groups(k, g):
    return (k + g - 1) // g


def _linear_inputs(case, seed):
    """(activations, stored weight arrays) on the GPU, from the seed."""
    g, m, k, n = _rng(seed), case["m"], case["k"], case["n"]
    a = _activations(g, m, k)
    if case["dtype"] == "i8":
        return a, [_i8(g, n, k), _f16_uniform(g, 1e-4, 3e-4, n).float()]
    scale = _f16_uniform(g, 4e-3, 8e-3, n, _groups(k, case["group"]))
    packed = _bytes(g, n, (k + 1) // 2)
    if case["dtype"] == "i4":
        return a, [packed, scale]
    return a, [packed, scale, (scale.float() * -7.5).half()]


def _moe_inputs(case, seed):
    """(x, router logits, {matrix: (weights, scales, mins)}) on the GPU; the
    matrices are stacked over the experts."""
    g, t, e, d, mi, dtype = _rng(seed), case["tokens"], case["experts"], case["d"], case["mi"], case["dtype"]
    x = torch.randn(t, d, generator=g, device="cuda")
    logits = torch.randn(t, e, generator=g, device="cuda")
    mats = {}
    for name, (i, o) in (("gate", (d, mi)), ("up", (d, mi)), ("down", (mi, d))):
        if dtype == "i8":
            mats[name] = (_i8(g, e, i, o), _f16_uniform(g, 2e-4, 4e-4, e, o), None)
        elif dtype == "f16":
            mats[name] = ((torch.randn(e, i, o, generator=g, device="cuda") * 0.02).half(), None, None)
        else:
            s = _f16_uniform(g, 4e-3, 8e-3, e, o, _groups(i, case["group"]))
            mats[name] = (_bytes(g, e, o, (i + 1) // 2), s, (s.float() * -7.5).half() if dtype == "q4a" else None)
    return x, logits, mats


def _write_bundle(case, seed):
    """A fresh folder with the case's bundle, and the bundle's stem."""
    arch, heads, kv, hd, d, ffn = FAMILIES[case["family"]]
    folder = tempfile.mkdtemp(prefix="frq_perf_", dir="/dev/shm" if os.path.isdir("/dev/shm") else None)
    stem = os.path.join(folder, "model")
    common = dict(n_layer=case["layers"], n_head=heads, n_kv=kv, hd=hd, d=d, ffn=ffn, vocab=case["vocab"],
                  dtype=case["dtype"])
    write = synth.write_rope_bundle if arch == "rope" else synth.write_gemma2_bundle
    write(stem, seed, raw=case["dtype"] == ("int8" if arch == "rope" else "int4"), **common)
    return folder, stem


def _prompts(case, seed):
    return np.stack([synth.gpt2_prompt(case["prompt"], case["vocab"], 1000 * seed + b) for b in range(case["batch"])])


def prepare(case, seed):
    ctx = _context()
    if case["kind"] == "linear":
        a, w = _linear_inputs(case, seed)
        host = [t.cpu().numpy() for t in w]
        if case["dtype"] == "i8":
            weight = ctx.upload_i8(*host)
        elif case["dtype"] == "i4":
            weight = ctx.upload_i4(*host, case["k"], case["group"])
        else:
            weight = ctx.upload_q4a(*host, case["k"], case["group"])
        call = {"mm": weight.mm_dev, "exact": weight.mm_exact_dev, "rows": weight.mm_rows_dev}[case["api"]]
        return {"kind": "linear", "weight": weight, "call": call, "a": a,
                "out": torch.empty(case["m"], case["n"], device="cuda")}
    if case["kind"] == "moe":
        x, logits, mats = _moe_inputs(case, seed)
        args = {}
        for name, (w, s, mn) in mats.items():
            args[name] = list(w.cpu().numpy().view(np.uint16) if case["dtype"] == "f16" else w.cpu().numpy())
            args[name + "_scale"] = None if s is None else list(_u16(s))
            args[name + "_min"] = None if mn is None else list(_u16(mn))
        bank = ctx.upload_moe(case["dtype"], case["d"], case["mi"], g=case.get("group", 0), **args)
        return {"kind": "moe", "bank": bank, "x": x, "logits": logits, "topk": case["topk"],
                "out": torch.empty(case["tokens"], case["d"], device="cuda")}
    folder, stem = _write_bundle(case, seed)
    try:
        bundle = fa.Bundle(stem, ctx)
        model = (fa.Rope if case["family"].startswith("rope") else fa.Gemma)(bundle, kv_int8=case["kv_int8"])
        bundle.close()
    finally:
        shutil.rmtree(folder, ignore_errors=True)
    return {"kind": "generate", "model": model, "prompts": _prompts(case, seed), "new": case["new"]}


def run(state):
    if state["kind"] == "linear":
        a, out = state["a"], state["out"]
        state["call"](a.data_ptr(), a.shape[0], out.data_ptr())
        return out
    if state["kind"] == "moe":
        x, out = state["x"], state["out"]
        state["bank"].forward_dev(x.data_ptr(), x.shape[0], state["logits"].data_ptr(), state["topk"], True, None,
                                  out.data_ptr())
        return out
    prompts = state["prompts"]
    if len(prompts) == 1:
        tokens, logits = state["model"].generate(prompts[0], state["new"], with_logits=True)
        return {"tokens": tokens, "first": logits[:1], "rest": logits[1:]}
    tokens, logits = state["model"].generate_batch(prompts, state["new"], with_logits=True)
    return {"tokens": tokens, "first": logits[:, 0], "rest": logits[:, 1:]}


def _weight_bytes(dtype, k, n, group=32):
    if dtype in ("i8", "int8"):
        return n * k + 4 * n
    if dtype in ("i4", "int4"):
        return n * ((k + 1) // 2) + 2 * n * _groups(k, group)
    if dtype == "q4a":
        return n * ((k + 1) // 2) + 4 * n * _groups(k, group)
    return 2 * n * k


def work(case):
    if case["kind"] == "linear":
        m, k, n = case["m"], case["k"], case["n"]
        return {"bytes": _weight_bytes(case["dtype"], k, n, case.get("group", 32)) + 4 * m * k + 4 * m * n,
                "flops": 2 * m * k * n}
    if case["kind"] == "moe":
        t, e, d, mi, top = (case[x] for x in ("tokens", "experts", "d", "mi", "topk"))
        active = e * (1.0 - (1.0 - top / e) ** t)
        per = 2 * _weight_bytes(case["dtype"], d, mi) + _weight_bytes(case["dtype"], mi, d)
        return {"bytes": int(active * per) + 8 * t * d + 4 * t * e, "flops": 6 * t * top * d * mi}
    _, heads, kv, hd, d, ffn = FAMILIES[case["family"]]
    shapes = [(d, (heads + 2 * kv) * hd), (heads * hd, d), (d, 2 * ffn), (ffn, d)]
    wide = case["layers"] * sum(k * n for k, n in shapes)
    held = case["layers"] * sum(_weight_bytes(case["dtype"], k, n) for k, n in shapes)
    steps, nb, p = case["new"] - 1, case["batch"], case["prompt"]
    head = case["vocab"] * d
    # the prompt's and each new token's linears, the causal half of the
    # scores and values, and one row of the head for each token chosen
    pairs = nb * (p * (p + 1) // 2 + sum(p + i for i in range(1, steps + 1)))
    flops = 2 * wide * nb * (p + steps) + 4 * case["layers"] * heads * hd * pairs + 2 * head * nb * case["new"]
    cache = case["layers"] * 2 * kv * hd * (1 if case["kv_int8"] else 4) * nb * sum(p + i for i in range(1, steps + 1))
    return {"bytes": (held + 2 * head) * case["new"] + cache + 4 * nb * case["new"] * case["vocab"], "flops": flops}


def tolerance(case):
    """Four times what another order of the 32-bit sums gives (measured
    against exact()); a generate call carries such a difference through the
    per-token int8 quantisation of every later layer, where one step of an
    int8 value or another outlier moves the logits far more."""
    if case["kind"] == "linear":
        return {"rel": 4e-6, "max": 1e-4}
    if case["kind"] == "moe":
        return {"rel": 4e-6, "max": 1e-4}
    int8 = case["dtype"] == "int8" or case["kv_int8"]
    return {"rel": 2e-2 if int8 else 1e-4, "max": 0.2 if int8 else 2e-3, "differ": 0.01}


# ---- the same values in 64 bits, by plain torch -----------------------------

def _quantise(a):
    """Per row of f32 a: (int8 values, step, outlier values in place)."""
    m, k = a.shape
    t = min(OUTLIERS, k)
    order = torch.sort(a.abs(), dim=1, descending=True, stable=True).indices
    out = torch.zeros_like(a, dtype=torch.bool).scatter_(1, order[:, :t], True)
    if t == k:
        sa = torch.ones(m, device=a.device)
    else:
        bulk = a.abs().gather(1, order[:, t:t + 1])[:, 0]
        sa = torch.where(bulk > 0, (bulk.double() / 127.0).float(), torch.ones_like(bulk))
    q = (a.double() / sa.double()[:, None]).float().double()
    q = (torch.sign(q) * torch.floor(q.abs() + 0.5)).clamp(-127, 127)
    return torch.where(out, 0.0, q), sa.double(), torch.where(out, a.double(), 0.0)


def _nibbles(packed, k, signed):
    q = torch.stack([packed & 15, packed >> 4], dim=-1).reshape(*packed.shape[:-1], -1)[..., :k].double()
    return torch.where(q >= 8, q - 16, q) if signed else q


def _dequant(dtype, w, s, mn, k, group):
    """(out, in) f64 of a stored int4 / q4a matrix."""
    rep = lambda v: v.double().repeat_interleave(group, dim=-1)[..., :k]
    if dtype in ("i4", "int4"):
        return _nibbles(w, k, True) * rep(s)
    return _nibbles(w, k, False) * rep(s) + rep(mn)


def _mm64(a, w, dtype, chunk=4096):
    """f32 / f64 rows a through a linear: w a f64 (out, in) matrix, or
    (int8 (out, in), scale) with the activations quantised a row at a time."""
    if dtype not in ("i8", "int8"):
        return a.double() @ w.T
    q, sa, ov = _quantise(a.float())
    wt, scale = w
    out = []
    for r in range(0, wt.shape[0], chunk):
        part = wt[r:r + chunk].double()
        out.append(scale[r:r + chunk].double() * (sa[:, None] * (q @ part.T) + ov @ part.T))
    return torch.cat(out, dim=1)


def _exact_moe(case, seed):
    x, logits, mats = _moe_inputs(case, seed)
    p = torch.softmax(logits.double(), dim=1)
    sel = torch.sort(p, dim=1, descending=True, stable=True).indices[:, :case["topk"]]
    wgt = p.gather(1, sel)
    wgt = wgt / wgt.sum(1, keepdim=True)
    out = torch.zeros(case["tokens"], case["d"], device="cuda", dtype=torch.float64)

    def mat(name, e):  # f64 (in, out)
        w, s, mn = mats[name]
        inp = case["mi"] if name == "down" else case["d"]
        if case["dtype"] == "i8":
            return w[e].double() * s[e].double()
        if case["dtype"] == "f16":
            return w[e].double()
        return _dequant(case["dtype"], w[e], s[e], None if mn is None else mn[e], inp, case["group"]).T

    for e in range(case["experts"]):
        tok, slot = torch.nonzero(sel == e, as_tuple=True)
        if len(tok):
            xe = x[tok].double()
            h = torch.nn.functional.silu(xe @ mat("gate", e)) * (xe @ mat("up", e))
            out.index_add_(0, tok, wgt[tok, slot][:, None] * (h @ mat("down", e)))
    return out


def _stored(stem):
    """{name: array} of a written bundle, as stored, with dtype and group."""
    import json
    with open(stem + ".fieldrun.json") as f:
        entries = json.load(f)["arrays"]
    blob = np.memmap(stem + ".fieldrun.bin", np.uint8, "r")
    kinds = {"f16": np.float16, "f32": np.float32, "i8": np.int8}
    got = {}
    for e in entries:
        raw = np.array(blob[e["offset"]:e["offset"] + e["bytes"]]).view(kinds.get(e["dtype"], np.uint8))
        shape = (e["shape"][0], -1) if e["dtype"] in ("i4", "q4a") else e["shape"]
        got[e["name"]] = (torch.from_numpy(raw.reshape(shape)).cuda(), e)
    return got


def _exact_generate(case, seed):
    """The logits after the prompt, of every sequence."""
    arch, heads, kv, hd, d, ffn = FAMILIES[case["family"]]
    folder, stem = _write_bundle(case, seed)
    try:
        arrays = _stored(stem)
    finally:
        shutil.rmtree(folder, ignore_errors=True)
    vec = lambda name: arrays[name][0].double()

    def linear(a, name):
        w, e = arrays[name]
        s = arrays[name + "__scale"][0]
        if e["dtype"] == "i8":
            return _mm64(a, (w.T, s), "int8")
        k = e["shape"][1]
        mn = arrays[name + "__min"][0] if e["dtype"] == "q4a" else None
        return _mm64(a, _dequant(e["dtype"], w, s, mn, k, e["group"]), e["dtype"])

    def norm(x, name):
        return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + 1e-6) * vec(name)

    def rope(x, n):  # (p, n * hd): halves rotated
        inv = 1.0 / (1e6 if arch == "rope" else 1e4) ** (torch.arange(0, hd, 2, device="cuda").double() / hd)
        ang = torch.arange(x.shape[0], device="cuda").double()[:, None] * inv
        c, s = ang.cos()[:, None], ang.sin()[:, None]
        x = x.view(-1, n, hd)
        lo, hi = x[..., :hd // 2], x[..., hd // 2:]
        return torch.cat([lo * c - hi * s, hi * c + lo * s], dim=-1)

    def cache(x):  # the int8 cache's values
        if not case["kv_int8"]:
            return x
        step = (x.abs().amax(-1, keepdim=True) / 127.0).clamp_min(1e-8)
        return (x / step).round().clamp(-127, 127) * step

    def logits_of(ids):
        x = vec("embed")[torch.from_numpy(ids).cuda()] * (math.sqrt(d) if arch == "gemma" else 1.0)
        p = len(ids)
        hidden = torch.ones(p, p, device="cuda", dtype=torch.bool).triu(1)
        for layer in range(case["layers"]):
            pre = "l%d." % layer
            h = norm(x, pre + ("input_layernorm" if arch == "gemma" else "in_ln"))
            q, k, v = (linear(h, pre + "self_attn." + t) for t in ("q_proj", "k_proj", "v_proj"))
            if arch == "rope":
                q, k, v = (t + vec(pre + "self_attn.%s_proj.bias" % b) for t, b in ((q, "q"), (k, "k"), (v, "v")))
            q, k, v = rope(q, heads), cache(rope(k, kv)), cache(v.view(p, kv, hd))
            att = torch.empty(p, heads, hd, device="cuda", dtype=torch.float64)
            for a in range(heads):
                s = q[:, a] @ k[:, a * kv // heads].T / math.sqrt(hd)
                if arch == "gemma":  # prompts are shorter than the sliding window
                    s = 50.0 * torch.tanh(s / 50.0)
                att[:, a] = torch.softmax(s.masked_fill(hidden, -1e30), -1) @ v[:, a * kv // heads]
            o = linear(att.view(p, -1), pre + "self_attn.o_proj")
            x = x + (norm(o, pre + "post_attention_layernorm") if arch == "gemma" else o)
            h = norm(x, pre + ("pre_feedforward_layernorm" if arch == "gemma" else "post_ln"))
            gate, up = linear(h, pre + "mlp.gate_proj"), linear(h, pre + "mlp.up_proj")
            act = torch.nn.functional.gelu(gate, approximate="tanh") if arch == "gemma" else \
                torch.nn.functional.silu(gate)
            o = linear(act * up, pre + "mlp.down_proj")
            x = x + (norm(o, pre + "post_feedforward_layernorm") if arch == "gemma" else o)
        return norm(x[-1:], "norm") @ vec("embed" if arch == "gemma" else "lm_head").T

    first = torch.cat([logits_of(ids) for ids in _prompts(case, seed)])
    return {"tokens": None, "first": first, "rest": None}


def exact(case, seed):
    if case["kind"] == "moe":
        return _exact_moe(case, seed)
    if case["kind"] == "generate":
        return _exact_generate(case, seed)
    a, w = _linear_inputs(case, seed)
    if case["dtype"] == "i8":
        return _mm64(a, w, "i8")
    mins = w[2] if case["dtype"] == "q4a" else None
    return _mm64(a, _dequant(case["dtype"], w[0], w[1], mins, case["k"], case["group"]), case["dtype"])
