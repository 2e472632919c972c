"""The workloads whose speed this framework is judged by: each is one call (or one short chain of calls) through the
public entry points, at sizes of the benchmark configurations (deepgengraph_amd/configs.py), of bench.py and of the
tests, together with the ranges around them.

    listed()             the named cases
    draw(rng)            one more case of the same ranges
    prepare(case, seed)  what a program holds before the call, on the GPU
    run(state)           one pass; its outputs
    work(case)           bytes and operations one pass cannot do without
    tolerance(case)      how far another correct implementation of the same precision may be
    exact(case, seed)    the outputs in 64 bits, in plain torch

Every case names its kind:

    prefill   causal attention over a prompt, optionally behind keys already in the cache (compile(Attn))
    gemma2    causal attention with grouped query heads, soft-cap and a sliding window, head_dim 256
    fp32      the same attention in fp32
    encoder   attention without a mask over a batch of sequences, head_dim 64
    decode    one decode step: RMSNorm and SiLU-and-mul of the step's rows, then one query row per sequence over
              its cache, in the cache layout [B, H, L, D] or the case layout [B, L, H, D] with grouped heads
    chunk     a few query rows (speculative decode, chunked prefill) over a long cache
    scores    the causal attention of the KV-selection cases with their key scores (H2O, RoCo, SnapKV, Corm)
    keyformer the same for KeyFormer, whose scores take a [B, H, S, S] random input
    compact   a selection from scores in hand and the gather of the kept rows of the cache
    block     the Llama attention block: RMSNorm, QKV projection, rotary, attention, output projection
"""
from __future__ import annotations

import math

import torch

from deepgengraph_amd import attention as A
from deepgengraph_amd import cases as C
from deepgengraph_amd import llama
from deepgengraph_amd.compile import compile as compile_case

_DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
_SIZE = {"f32": 4, "f16": 2, "bf16": 2}
_EPS = 1e-6
_THETA = 10000.0


def listed():
    return [
        # Llama-2-7B prefill of a 4096-token prompt: the benchmark's headline workload.
        dict(name="prefill_7b", kind="prefill", B=1, S=4096, past=0, H=32, Hkv=32, D=128, dtype="bf16"),
        # A short chat turn, of no round length: latency and a chip that few workgroups fill.
        dict(name="prefill_short", kind="prefill", B=1, S=509, past=0, H=32, Hkv=32, D=128, dtype="bf16"),
        # Gemma-2 attention at its full context: grouped heads, soft-cap, sliding window.
        dict(name="prefill_gemma2", kind="gemma2", B=2, S=8192, H=16, Hkv=8, D=256, softcap=50.0, window=4096,
             dtype="bf16"),
        # The fp32 configuration, used to check a model in full precision: the smallest attention call.
        dict(name="prefill_fp32", kind="fp32", B=1, S=512, H=8, D=64, dtype="f32"),
        # An encoder batch: no mask, small heads, sequences of no round length.
        dict(name="encoder_d64", kind="encoder", B=8, S=1000, H=16, D=64, dtype="f16"),
        # Batch serving with long contexts: the decode benchmark (34 GB of cache).
        dict(name="decode_7b", kind="decode", layout="cache", B=64, L=32768, H=32, Hkv=32, D=128, hidden=4096,
             inter=11008, dtype="f16"),
        # One user's chat: one sequence, grouped heads, a cache of no round length. Launches and latency count.
        dict(name="decode_gqa", kind="decode", layout="case", B=1, L=4001, H=32, Hkv=8, D=128, hidden=4096,
             inter=14336, dtype="bf16"),
        # Verification of 16 drafted tokens over a 32K context.
        dict(name="chunk_32k", kind="chunk", B=1, q=16, L=32768, H=32, Hkv=32, D=128, dtype="f16"),
        # H2O's prefill: attention and the column sums its cache selection ranks keys by.
        dict(name="scores_h2o", kind="scores", policy="h2o", B=1, S=4096, H=32, D=128, dtype="f16"),
        # KeyFormer's prefill at half that length (its random input alone is B*H*S*S floats).
        dict(name="scores_keyformer", kind="keyformer", B=1, S=2048, H=32, D=128, dtype="f16"),
        # The cache cut down after a 128K-token prompt.
        dict(name="compact_128k", kind="compact", B=1, S=131072, H=32, D=128, k=256, dtype="f16"),
        # A whole attention block, with its projections.
        dict(name="block_7b", kind="block", B=1, S=4096, H=32, Hkv=32, D=128, dtype="bf16"),
    ]


def _log(rng, lo, hi):
    """A whole number of [lo, hi], evenly over its logarithm; half of them made multiples of 64 where that fits."""
    x = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if x > 128 and rng.random() < 0.5:
        x -= x % 64
    return max(lo, min(hi, x))


def draw(rng):
    kind = rng.choice(["prefill", "prefill", "gemma2", "fp32", "encoder", "decode", "decode", "chunk", "scores",
                       "keyformer", "compact", "block"])
    half = rng.choice(["f16", "bf16"])
    if kind == "prefill":
        B = rng.choice([1, 1, 2, 4])
        S = _log(rng, 64, 8192 // B)
        past = rng.choice([0, 0, 0, _log(rng, 64, 4096)]) if S <= 4096 else 0
        return dict(kind=kind, B=B, S=S, past=past, H=32, Hkv=rng.choice([32, 32, 8]), D=128, dtype=half)
    if kind == "gemma2":
        return dict(kind=kind, B=rng.choice([1, 2]), S=_log(rng, 256, 8192), H=16, Hkv=8, D=256, softcap=50.0,
                    window=4096, dtype="bf16")
    if kind == "fp32":
        return dict(kind=kind, B=rng.choice([1, 2]), S=_log(rng, 64, 1024), H=8, D=rng.choice([64, 128]), dtype="f32")
    if kind == "encoder":
        B = _log(rng, 1, 16)
        return dict(kind=kind, B=B, S=_log(rng, 64, 2048), H=rng.choice([12, 16]), D=64, dtype=half)
    if kind == "decode":
        B, L = _log(rng, 1, 64), _log(rng, 128, 32768)
        if rng.random() < 0.5:
            return dict(kind=kind, layout="cache", B=B, L=L, H=32, Hkv=32, D=128, hidden=4096, inter=11008, dtype=half)
        return dict(kind=kind, layout="case", B=B, L=L, H=32, Hkv=8, D=128, hidden=4096, inter=14336, dtype=half)
    if kind == "chunk":
        return dict(kind=kind, B=rng.choice([1, 2]), q=_log(rng, 2, 64), L=_log(rng, 2048, 65536), H=32,
                    Hkv=rng.choice([32, 8]), D=128, dtype=half)
    if kind == "scores":
        return dict(kind=kind, policy=rng.choice(["h2o", "roco", "snapkv", "corm"]), B=rng.choice([1, 1, 2]),
                    S=_log(rng, 256, 4096), H=32, D=128, dtype=half)
    if kind == "keyformer":
        return dict(kind=kind, B=1, S=_log(rng, 256, 4096), H=32, D=128, dtype=half)
    if kind == "compact":
        S = _log(rng, 512, 131072)
        return dict(kind=kind, B=1, S=S, H=rng.choice([8, 32]), D=128, k=_log(rng, 64, min(2048, S // 2)), dtype=half)
    return dict(kind="block", B=rng.choice([1, 2]), S=_log(rng, 64, 4096), H=32, Hkv=rng.choice([32, 8]), D=128,
                dtype="bf16")


# --------------------------------------------------------------------------------------------------------------------
# Inputs
# --------------------------------------------------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _randn(g, dtype, *shape, mean=0.0, std=1.0):
    return (torch.randn(*shape, generator=g, device="cuda") * std + mean).to(dtype)


def _qkv(case, g, Sq, Sk, Hkv):
    dt = _DTYPES[case["dtype"]]
    q = _randn(g, dt, case["B"], Sq, case["H"], case["D"])
    return q, _randn(g, dt, case["B"], Sk, Hkv, case["D"]), _randn(g, dt, case["B"], Sk, Hkv, case["D"])


def _inputs(case, seed):
    """The tensors of a case, from the seed alone."""
    g, kind, dt = _gen(seed), case["kind"], _DTYPES[case["dtype"]]
    B, H, D = case["B"], case["H"], case["D"]
    if kind == "prefill":
        q, k, v = _qkv(case, g, case["S"], case["S"] + case["past"], case["Hkv"])
        return dict(q=q, k=k, v=v)
    if kind == "gemma2":
        q, k, v = _qkv(case, g, case["S"], case["S"], case["Hkv"])
        return dict(q=q, k=k, v=v)
    if kind in ("fp32", "encoder"):
        q, k, v = _qkv(case, g, case["S"], case["S"], H)
        return dict(q=q, k=k, v=v)
    if kind == "chunk":
        q, k, v = _qkv(case, g, case["q"], case["L"], case["Hkv"])
        return dict(q=q, k=k, v=v)
    if kind == "decode":
        s = dict(x=_randn(g, dt, B, case["hidden"]), w=_randn(g, dt, case["hidden"], mean=1.0, std=0.02),
                 gate_up=_randn(g, dt, B, 2 * case["inter"]))
        if case["layout"] == "cache":
            s["q"] = _randn(g, dt, B, H, D)
            shape = (case["Hkv"], case["L"], D)
        else:
            s["q"] = _randn(g, dt, B, 1, H, D)
            shape = (case["L"], case["Hkv"], D)
        for name in ("k", "v"):  # one sequence at a time: no fp32 copy of the whole cache
            s[name] = torch.empty(B, *shape, dtype=dt, device="cuda")
            for b in range(B):
                s[name][b] = torch.randn(*shape, generator=g, device="cuda", dtype=dt)
        return s
    if kind in ("scores", "keyformer"):
        S = case["S"]
        q, k, v = _qkv(case, g, S, S, H)
        # heavy hitters: 16 keys of four times the length (as the H2O configuration draws them)
        k[:, torch.randperm(S, generator=g, device="cuda")[:16]] *= 4.0
        s = dict(q=q, k=k, v=v)
        if case.get("policy") == "corm":  # row i of the thresholds is 1 / (i + 1)
            s["mask"] = (1.0 / torch.arange(1, S + 1, dtype=torch.float32, device="cuda")).unsqueeze(1).expand(
                S, S).contiguous()
        if kind == "keyformer":
            s["rand"] = torch.randn(B, H, S, S, generator=g, device="cuda").abs_().add_(1.0)
        return s
    if kind == "compact":
        S = case["S"]
        # scores as column sums of a causal softmax have them: positive, larger for early keys
        score = torch.rand(B, H, S, generator=g, device="cuda") * (
            1.0 + 50.0 / (1.0 + torch.arange(S, device="cuda", dtype=torch.float32).sqrt()))
        return dict(score=score, k=_randn(g, dt, B, S, H, D), v=_randn(g, dt, B, S, H, D))
    hidden, kv = H * D, case["Hkv"] * D
    return dict(x=_randn(g, dt, B, case["S"], hidden), w_norm=_randn(g, dt, hidden, mean=1.0, std=0.02),
                w_qkv=_randn(g, dt, hidden + 2 * kv, hidden, std=0.02), w_o=_randn(g, dt, hidden, hidden, std=0.02))


_POLICY = {"h2o": C.H2O, "roco": C.RoCo, "snapkv": C.SnapKV, "corm": C.Corm}


def prepare(case, seed):
    s = _inputs(case, seed)
    s["case"] = dict(case)
    kind, H, D = case["kind"], case["H"], case["D"]
    if kind in ("prefill", "fp32"):
        model = C.Attn(kv_head_num=H, head_num=H, head_dim=D)
        s["f"] = compile_case(model, ["q", "k", "v"], [s["q"], s["k"], s["v"]], ["out"], "mi355x")
    elif kind == "scores":
        model = _POLICY[case["policy"]](kv_head_num=H, head_num=H, head_dim=D)
        s["args"] = [s["q"], s["k"], s["v"]] + ([s["mask"]] if "mask" in s else [])
        names = ["q", "k", "v"] + (["corm_mask"] if "mask" in s else [])
        s["f"] = compile_case(model, names, s["args"], list(model.OUTPUTS), "mi355x")
    elif kind == "keyformer":
        model = C.KeyFormer(kv_head_num=H, head_num=H, head_dim=D)
        s["f"] = compile_case(model, ["q", "k", "v", "exp_rand"], [s["q"], s["k"], s["v"], s["rand"]],
                              list(model.OUTPUTS), "mi355x")
    elif kind == "block":
        s["f"] = llama.LlamaAttentionBlock(s["w_norm"], s["w_qkv"], s["w_o"], heads=H, kv_heads=case["Hkv"], eps=_EPS,
                                           rope_theta=_THETA)
    return s


# --------------------------------------------------------------------------------------------------------------------
# One pass
# --------------------------------------------------------------------------------------------------------------------
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind in ("prefill", "fp32"):
        return state["f"](state["q"], state["k"], state["v"])
    if kind == "gemma2":
        return A.attention(state["q"], state["k"], state["v"], causal=True, softcap=case["softcap"],
                           window=case["window"])
    if kind == "encoder":
        return A.attention(state["q"], state["k"], state["v"], causal=False)
    if kind == "decode":
        normed, act = llama.decode_prestep(state["x"], state["w"], state["gate_up"], _EPS)
        if case["layout"] == "cache":
            out = A.decode_attention(state["q"], state["k"], state["v"])
        else:
            out = A.attention(state["q"], state["k"], state["v"])
        return normed, act, out
    if kind == "chunk":
        return A.attention(state["q"], state["k"], state["v"], causal=True)
    if kind == "scores":
        return state["f"](*state["args"])
    if kind == "keyformer":
        return state["f"](state["q"], state["k"], state["v"], state["rand"])
    if kind == "compact":
        keep = A.topk_indices(state["score"], case["k"])
        return keep, A.kv_gather(state["k"], state["v"], keep)
    return state["f"](state["x"])


# --------------------------------------------------------------------------------------------------------------------
# What a pass cannot do without
# --------------------------------------------------------------------------------------------------------------------
def _pairs(Sq, Sk, window=0):
    """Visible (query, key) pairs of a causal head."""
    total, off = 0, Sk - Sq
    for i in range(Sq):
        total += min(Sk, i + off + 1) - (max(0, i + off - window + 1) if window else 0)
    return total


def work(case):
    kind, B, H, D, e = case["kind"], case["B"], case["H"], case["D"], _SIZE[case["dtype"]]
    Hkv = case.get("Hkv", H)

    def attn(Sq, Sk, pairs):
        return (e * B * D * (2 * Sq * H + 2 * Sk * Hkv), 4.0 * D * B * H * pairs)

    if kind == "prefill":
        by, fl = attn(case["S"], case["S"] + case["past"], _pairs(case["S"], case["S"] + case["past"]))
    elif kind == "gemma2":
        by, fl = attn(case["S"], case["S"], _pairs(case["S"], case["S"], case["window"]))
    elif kind == "fp32":
        by, fl = attn(case["S"], case["S"], _pairs(case["S"], case["S"]))
    elif kind == "encoder":
        by, fl = attn(case["S"], case["S"], case["S"] ** 2)
    elif kind == "chunk":
        by, fl = attn(case["q"], case["L"], _pairs(case["q"], case["L"]))
    elif kind == "decode":
        by, fl = attn(1, case["L"], case["L"])
        by += e * (2 * B * case["hidden"] + case["hidden"] + 3 * B * case["inter"])
        fl += B * (4.0 * case["hidden"] + 6.0 * case["inter"])
    elif kind in ("scores", "keyformer"):
        S = case["S"]
        by, fl = attn(S, S, _pairs(S, S))
        by += 4 * B * H * S * (2 if case.get("policy") == "roco" else 1)
        # the scores need every row's normaliser before any column can be summed: the products again, or stored
        fl += 2.0 * D * B * H * _pairs(S, S)
        if case.get("policy") == "corm":
            by += 4 * S * S - 3 * B * H * S
        if kind == "keyformer":
            by += 4 * B * H * _pairs(S, S)
    elif kind == "compact":
        rows = B * H
        by = rows * (4 * case["S"] + 8 * case["k"] + 2 * 2 * e * case["k"] * D)
        fl = float(rows * case["S"])
    else:
        hidden, kv, T = H * D, Hkv * D, B * case["S"]
        by = e * (2 * T * hidden + hidden + (hidden + 2 * kv) * hidden + hidden * hidden)
        fl = 2.0 * T * hidden * (2 * hidden + 2 * kv) + 4.0 * D * B * H * _pairs(case["S"], case["S"])
    return {"bytes": int(by), "flops": float(fl)}


# --------------------------------------------------------------------------------------------------------------------
# How far another correct implementation may be, and the 64-bit results
# --------------------------------------------------------------------------------------------------------------------
def tolerance(case):
    """About four times the error of these calls against exact(), which is that of the results' rounding to their type:
    2.9e-4 for f16 and 2.6e-3 for bf16; 2.5e-7 for the fp32 call (its 32-bit sums and exponentials). A block's four
    roundings in a row (normalised rows, q/k/v, attention, projection) leave 8.6e-3."""
    kind = case["kind"]
    if kind == "compact":
        return "exact"
    if kind == "fp32":
        return {"rel": 2e-6}
    if kind == "block":
        return {"rel": 2e-2}
    tol = {"rel": 1.2e-3 if case["dtype"] == "f16" else 1e-2}
    if case.get("policy") == "corm":
        tol["differ"] = 1e-3  # probabilities that equal their threshold but for the last bit
    return tol


def _attn64(q, k, v, *, causal=True, softcap=0.0, window=0, rounded=None, extra=None):
    """Attention of q [B, Sq, H, D] over k, v [B, Sk, Hkv, D] in 64 bits, some heads at a time; the output as
    [B, Sq, H, D]. rounded: the 16-bit type the scores are rounded to where the reference's module rounds them (the
    product, then the product over sqrt(D)). extra(b, h, scores, probs) sees each head's [Sq, Sk] matrices."""
    B, Sq, H, D = q.shape
    Sk, group = k.shape[1], H // k.shape[2]
    out = torch.empty(B, Sq, H, D, dtype=torch.float64, device=q.device)
    i = torch.arange(Sq, device=q.device).unsqueeze(1) + (Sk - Sq)
    j = torch.arange(Sk, device=q.device).unsqueeze(0)
    hidden = torch.zeros(Sq, Sk, dtype=torch.bool, device=q.device)
    if causal:
        hidden |= j > i
    if window:
        hidden |= j <= i - window
    for b in range(B):
        for h in range(H):
            kh, vh = (t[b, :, h // group].double() for t in (k, v))
            s = torch.mm(q[b, :, h].double(), kh.t().contiguous())
            if rounded is not None:
                s = s.to(rounded)
                s = (s.float() * torch.tensor(1.0 / math.sqrt(D), device=q.device)).to(rounded).double()
            else:
                s /= math.sqrt(D)
            if softcap:
                s = softcap * torch.tanh(s / softcap)
            s.masked_fill_(hidden, -math.inf)
            p = torch.softmax(s, dim=-1)
            out[b, :, h] = torch.mm(p, vh)
            if extra is not None:
                extra(b, h, s, p)
    return out


def _norm64(x, w):
    x = x.double()
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + _EPS) * w.double()


def exact(case, seed):
    kind = case["kind"]
    s = _inputs(case, seed)
    if kind in ("prefill", "fp32", "chunk"):
        return _attn64(s["q"], s["k"], s["v"])
    if kind == "gemma2":
        return _attn64(s["q"], s["k"], s["v"], softcap=case["softcap"], window=case["window"])
    if kind == "encoder":
        return _attn64(s["q"], s["k"], s["v"], causal=False)
    if kind == "decode":
        q, k, v = s["q"], s["k"], s["v"]
        normed = _norm64(s["x"], s["w"])
        gate, up = s["gate_up"].double().chunk(2, dim=-1)
        act = torch.nn.functional.silu(gate) * up
        out = torch.empty(q.shape, dtype=torch.float64, device=q.device)
        group = case["H"] // case["Hkv"]
        for b in range(case["B"]):
            for hk in range(case["Hkv"]):
                hs = slice(hk * group, (hk + 1) * group)
                kc, vc = (t[b, hk] if case["layout"] == "cache" else t[b, :, hk] for t in (k, v))
                qh = (q[b, hs] if case["layout"] == "cache" else q[b, 0, hs]).double()
                p = torch.softmax(torch.mm(qh, kc.double().t().contiguous()) / math.sqrt(case["D"]), dim=-1)
                o = torch.mm(p, vc.double())
                if case["layout"] == "cache":
                    out[b, hs] = o
                else:
                    out[b, 0, hs] = o
        return normed, act, out
    if kind in ("scores", "keyformer"):
        B, H, S = case["B"], case["H"], case["S"]
        dt = _DTYPES[case["dtype"]]
        s1 = torch.zeros(B, H, S, dtype=torch.float64, device="cuda")
        s2 = torch.zeros_like(s1)
        hit = torch.zeros(B, H, S, dtype=torch.bool, device="cuda")
        policy = case.get("policy", "keyformer")

        def extra(b, h, scores, p):
            if policy == "corm":
                hit[b, h] = (p >= s["mask"]).any(0)
            elif policy == "keyformer":
                s1[b, h] = torch.softmax((scores - s["rand"][b, h].double().log()) / 1.5, dim=-1).sum(0)
            else:
                s1[b, h] = p.sum(0)
                s2[b, h] = (p * p).sum(0)

        out = _attn64(s["q"], s["k"], s["v"], rounded=dt, extra=extra)
        if policy == "corm":
            return out, hit
        if policy == "roco":
            return out, s1, s2
        if policy == "snapkv":
            return out, torch.nn.functional.avg_pool1d(s1, 5, stride=1, padding=2)
        return out, s1
    if kind == "block":
        B, S, H, Hkv, D = case["B"], case["S"], case["H"], case["Hkv"], case["D"]
        qkv = torch.matmul(_norm64(s["x"], s["w_norm"]), s["w_qkv"].double().t().contiguous())
        q, k, v = (t.view(B, S, -1, D) for t in qkv.split([H * D, Hkv * D, Hkv * D], dim=-1))
        ang = torch.arange(S, device="cuda").double().unsqueeze(1) * _THETA ** (
            -torch.arange(0, D, 2, device="cuda").double() / D)
        cos, sin = ang.cos().view(1, S, 1, D // 2), ang.sin().view(1, S, 1, D // 2)

        def rot(t):
            a, b = t[..., : D // 2], t[..., D // 2:]
            return torch.cat([a * cos - b * sin, b * cos + a * sin], dim=-1)

        o = _attn64(rot(q), rot(k), v)
        return torch.matmul(o.view(B, S, H * D), s["w_o"].double().t().contiguous())
    return None
