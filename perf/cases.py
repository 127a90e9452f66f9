"""The work that programs have this package do, as measurable cases: decode
steps of the persistent kernel, the fused operators at decode and at prompt
sizes, paged and causal attention, and kernel graphs through superoptimize.

Sizes are those of a Llama-3-8B-shaped model (hidden 4096, 32 / 8 heads of
128, MLP 14336, vocabulary 128256) and of the benchmark graphs under tests/;
draw() spreads rows, lengths, layouts, head counts and types around them.
"""
import math

import numpy as np
import torch

import yirage_amd as yr
from yirage_amd import fused
from yirage_amd.llama import LlamaConfig, LlamaDecodeModel

NK, KN = 0, 1  # weight layouts: [N, K] (torch Linear.weight) and [K, N] (x @ W)
DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16}
VOCAB = 128256


def listed():
    return [
        # one decode step of one conversation, 4 K tokens in: the headline step
        # (8 of its 32 layers, the LM head and the argmax)
        {"name": "step_b1", "kind": "step", "layers": 8, "rows": 1, "kv": 4096},
        # the same step for a batch of eight conversations (packed weights)
        {"name": "step_b8", "kind": "step", "layers": 4, "rows": 8, "kv": 4096},
        # the smallest call: the RMSNorm + projection kernel graph of a decode
        # batch, as superoptimize() returns it
        {"name": "graph_norm_proj_b8", "kind": "graph_norm", "rows": 8, "k": 4096, "n": 4096, "dtype": "f16"},
        # gated MLP of a decode batch: the weight stream
        {"name": "mlp_b8", "kind": "mlp", "rows": 8, "k": 4096, "n": 14336, "layout": KN, "dtype": "bf16"},
        # gated MLP of a large serving batch
        {"name": "mlp_b128", "kind": "mlp", "rows": 128, "k": 4096, "n": 14336, "layout": KN, "dtype": "bf16"},
        # gated MLP over a 2048-token prompt: the largest product of a prefill
        {"name": "mlp_prompt_2048", "kind": "mlp", "rows": 2048, "k": 4096, "n": 14336, "layout": KN,
         "dtype": "bf16"},
        # RMSNorm + QKV projection of a prompt of no round length, with the
        # checkpoint's own [N, K] weights
        {"name": "norm_qkv_prompt_777", "kind": "rms", "rows": 777, "k": 4096, "n": 6144, "layout": NK,
         "dtype": "bf16"},
        # down projection with the residual of a single token, [N, K] weights
        {"name": "down_residual_b1", "kind": "linear", "rows": 1, "k": 14336, "n": 4096, "layout": NK,
         "residual": True, "dtype": "f16"},
        # LM head and greedy token choice of a decode batch
        {"name": "head_argmax_b8", "kind": "head", "rows": 8, "k": 4096, "n": VOCAB, "dtype": "bf16"},
        # paged attention of a decode batch whose sequences differ in length
        {"name": "paged_decode_b8", "kind": "decode", "rows": 8, "hq": 32, "hkv": 8, "kv": 4096, "page": 64,
         "dtype": "f16"},
        # causal attention over a 2048-token prompt
        {"name": "prefill_2048", "kind": "prefill", "rows": 1, "seq": 2048, "hq": 32, "hkv": 8, "causal": True,
         "dtype": "bf16"},
        # the grouped-query attention benchmark graph (batch 8, head dim 64, K
        # given as [g, d, l]), as superoptimize() returns it
        {"name": "graph_gqa_bs8", "kind": "graph_attn", "rows": 16, "m": 256, "kv": 4096, "d": 64, "dtype": "f16"},
    ]


def _log(rng, lo, hi, step=1):
    """An integer spread over the logarithm of [lo, hi], a multiple of step."""
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / step)) * step
    return max(lo, min(hi, v))


def draw(rng):
    kind = rng.choice(["step", "graph_norm", "mlp", "mlp", "rms", "linear", "linear", "head", "decode", "prefill",
                       "graph_attn"])
    dtype = rng.choice(["f16", "bf16"])
    if kind == "step":
        return {"kind": kind, "layers": rng.randint(1, 4), "rows": _log(rng, 1, 16), "kv": _log(rng, 64, 4096)}
    if kind == "graph_norm":
        return {"kind": kind, "rows": _log(rng, 1, 128), "k": _log(rng, 512, 8192, 8), "n": _log(rng, 512, 8192, 8),
                "dtype": dtype}
    if kind == "mlp":
        return {"kind": kind, "rows": _log(rng, 1, 2048), "k": _log(rng, 1024, 4096, 8),
                "n": _log(rng, 1024, 14336, 8), "layout": rng.choice([NK, KN]), "dtype": dtype}
    if kind == "rms":
        return {"kind": kind, "rows": _log(rng, 1, 2048), "k": _log(rng, 1024, 8192, 8),
                "n": _log(rng, 1024, 14336, 8), "layout": rng.choice([NK, KN]), "dtype": dtype}
    if kind == "linear":
        return {"kind": kind, "rows": _log(rng, 1, 2048), "k": _log(rng, 1024, 14336, 8),
                "n": _log(rng, 1024, 8192, 8), "layout": rng.choice([NK, KN]), "residual": rng.random() < 0.5,
                "dtype": dtype}
    if kind == "head":
        return {"kind": kind, "rows": _log(rng, 1, 32), "k": _log(rng, 1024, 4096, 8),
                "n": _log(rng, 32000, VOCAB, 8), "dtype": dtype}
    if kind == "decode":
        hkv = rng.choice([2, 4, 8, 16])
        return {"kind": kind, "rows": _log(rng, 1, 32), "hq": hkv * rng.choice([1, 2, 4, 8]), "hkv": hkv,
                "kv": _log(rng, 64, 8192), "page": rng.choice([16, 64, 128]), "dtype": dtype}
    if kind == "prefill":
        hkv = rng.choice([4, 8])
        return {"kind": kind, "rows": rng.randint(1, 2), "seq": _log(rng, 64, 3072), "hq": hkv * rng.choice([1, 4]),
                "hkv": hkv, "causal": rng.random() < 0.75, "dtype": dtype}
    return {"kind": kind, "rows": _log(rng, 2, 32), "m": rng.choice([1, 4, 16, 64, 256]), "kv": _log(rng, 256, 4096, 8),
            "d": rng.choice([64, 128]), "dtype": dtype}


# ------------------------------------------------------------------ inputs
def _normal(gen, shape, std, dtype):
    return torch.empty(shape, dtype=dtype, device="cuda").normal_(0.0, std, generator=gen)


def _gamma(gen, n, dtype):
    return (1.0 + torch.empty(n, device="cuda").normal_(0.0, 0.1, generator=gen)).to(dtype)


def _dense(case, seed):
    """Activations, norm weight, weight(s) and residual of an operator call."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dt, B, K, N = DTYPES[case["dtype"]], case["rows"], case["k"], case["n"]
    kind = case["kind"]
    wshape = (K, N) if kind == "graph_norm" or case.get("layout", NK) == KN else (N, K)
    t = {"x": _normal(gen, (B, K), 1.0, dt)}
    if kind == "rms":
        t["gamma"] = _gamma(gen, K, dt)
    t["w"] = _normal(gen, wshape, 0.02, dt)
    if kind == "mlp":
        t["w3"] = _normal(gen, wshape, 0.02, dt)
    if kind == "head":
        t["w"].mul_(_head_scale(gen, N).to(dt))
    if case.get("residual"):
        t["residual"] = _normal(gen, (B, N), 1.0, dt)
    return t


def _head_scale(gen, n):
    """Row norms of a trained LM head differ; the likely tokens stand apart."""
    return torch.empty((n, 1), device="cuda").normal_(0.0, 0.4, generator=gen).exp()


def _paged(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    rng = np.random.default_rng(seed)
    dt, B, L, page = DTYPES[case["dtype"]], case["rows"], case["kv"], case["page"]
    # a batch in service: the longest sequence has L tokens, the others half to all of that
    lens = rng.integers((L + 1) // 2, L + 1, size=B)
    lens[rng.integers(B)] = L
    npg = -(-lens // page)
    pool = int(npg.sum())
    kv = (pool, page, case["hkv"], 128)
    return {"q": _normal(gen, (B, case["hq"], 128), 1.0, dt), "k": _normal(gen, kv, 1.0, dt),
            "v": _normal(gen, kv, 1.0, dt),
            "indptr": torch.from_numpy(np.concatenate([[0], np.cumsum(npg)]).astype(np.int32)).cuda(),
            "indices": torch.from_numpy(rng.permutation(pool).astype(np.int32)).cuda(),
            "lens": torch.from_numpy(lens.astype(np.int32)).cuda()}


def _prompt(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dt, B, S = DTYPES[case["dtype"]], case["rows"], case["seq"]
    return {"q": _normal(gen, (B, S, case["hq"], 128), 1.0, dt), "k": _normal(gen, (B, S, case["hkv"], 128), 1.0, dt),
            "v": _normal(gen, (B, S, case["hkv"], 128), 1.0, dt)}


def _graph_attn(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dt, G, M, L, d = DTYPES[case["dtype"]], case["rows"], case["m"], case["kv"], case["d"]
    # the graph has no softmax scale: its operands carry it
    std = d ** -0.25
    return {"q": _normal(gen, (G, M, d), std, dt), "k": _normal(gen, (G, d, L), std, dt),
            "v": _normal(gen, (G, L, d), 1.0, dt)}


def _config(case):
    return LlamaConfig(num_layers=case["layers"])


def _checkpoint(case, seed):
    """The tensors of a step, one at a time, in a fixed order: (layer or None,
    name, values); a program copies them into the model."""
    cfg, page = _config(case), 64
    gen = torch.Generator(device="cuda").manual_seed(seed)
    bf, h, d = torch.bfloat16, cfg.hidden, cfg.head_dim
    shapes = {"wq": (cfg.num_q_heads * d, h), "wk": (cfg.num_kv_heads * d, h), "wv": (cfg.num_kv_heads * d, h),
              "wo": (h, cfg.num_q_heads * d), "wg": (cfg.intermediate, h), "wu": (cfg.intermediate, h),
              "wd": (h, cfg.intermediate)}
    pool = case["rows"] * -(-case["kv"] // page)
    yield None, "embed", _normal(gen, (cfg.vocab, h), cfg.weight_std, bf)
    for layer in range(cfg.num_layers):
        for name, shape in shapes.items():
            yield layer, name, _normal(gen, shape, cfg.weight_std, bf)
        yield layer, "ln1", _gamma(gen, h, bf)
        yield layer, "ln2", _gamma(gen, h, bf)
        yield layer, "k", _normal(gen, (pool, page, cfg.num_kv_heads, d), 1.0, bf)
        yield layer, "v", _normal(gen, (pool, page, cfg.num_kv_heads, d), 1.0, bf)
    yield None, "norm", _gamma(gen, h, bf)
    head = _normal(gen, (cfg.vocab, h), cfg.weight_std, bf)
    yield None, "lm_head", head.mul_(_head_scale(gen, cfg.vocab).to(bf))


def _tokens_and_pages(case, seed):
    rng = np.random.default_rng(seed)
    pool = case["rows"] * -(-case["kv"] // 64)
    return rng.integers(0, VOCAB, size=case["rows"]), rng.permutation(pool).astype(np.int32)


def _model(case, seed):
    m = LlamaDecodeModel(_config(case), batch=case["rows"], kv_len=case["kv"], seed=0)
    whole = {"embed": m.embed, "norm": m.final_norm, "lm_head": m.lm_head}
    for layer, name, values in _checkpoint(case, seed):
        if layer is None:
            to = whole[name]
        else:
            to = m.kc[layer] if name == "k" else m.vc[layer] if name == "v" else m.w[layer][name]
        to.copy_(values)
    ids, pages = _tokens_and_pages(case, seed)
    m.meta["paged_kv_indices_buffer"].copy_(torch.from_numpy(pages))
    m.set_input_tokens(ids)
    if case["rows"] > 1:
        m.pk.pack_weights()  # the weights changed after compile
    return m


def prepare(case, seed):
    kind = case["kind"]
    if kind == "step":
        return {"case": case, "model": _model(case, seed)}
    if kind in ("graph_norm", "graph_attn"):
        dt = yr.float16 if case["dtype"] == "f16" else yr.bfloat16
        g = yr.new_kernel_graph()
        if kind == "graph_norm":
            t = _dense(case, seed)
            x, w = (g.new_input(dims=tuple(t[n].shape), dtype=dt) for n in ("x", "w"))
            g.mark_output(g.matmul(g.rms_norm(x, normalized_shape=(case["k"],)), w))
            inputs = [t["x"], t["w"]]
        else:
            t = _graph_attn(case, seed)
            q, k, v = (g.new_input(dims=tuple(t[n].shape), dtype=dt) for n in ("q", "k", "v"))
            e = g.exp(g.matmul(q, k))
            g.mark_output(g.matmul(g.div(e, g.reduction(e, 2)), v))
            inputs = [t["q"], t["k"], t["v"]]
        return {"case": case, "graph": g.superoptimize(backend="hip", warmup_iters=4, profile_iters=16),
                "inputs": inputs}
    make = {"decode": _paged, "prefill": _prompt}.get(kind, _dense)
    return {"case": case, **make(case, seed)}


# ------------------------------------------------------------------ one pass
def run(s):
    c = s["case"]
    kind = c["kind"]
    if kind == "step":
        m = s["model"]
        m.step()
        return {"logits": m.t["argmax_in"].tensor, "tokens": m.meta["output_tokens"], "k": m.kc, "v": m.vc}
    if kind in ("graph_norm", "graph_attn"):
        return s["graph"](inputs=s["inputs"])
    if kind == "mlp":
        return fused.gated_mlp(s["x"], s["w"], s["w3"], w_layout=c["layout"])
    if kind == "rms":
        return fused.rmsnorm_linear(s["x"], s["gamma"], s["w"], w_layout=c["layout"])
    if kind == "linear":
        return fused.linear(s["x"], s["w"], residual=s.get("residual"), w_layout=c["layout"])
    if kind == "head":
        logits = fused.linear(s["x"], s["w"])
        return logits, fused.argmax(logits)
    if kind == "decode":
        return fused.gqa_decode_paged(s["q"], s["k"], s["v"], s["indptr"], s["indices"], s["lens"],
                                      max_kv_len=c["kv"])
    return fused.gqa_prefill(s["q"], s["k"], s["v"], causal=c["causal"])


def work(case):
    kind, B = case["kind"], case["rows"]
    if kind == "step":
        cfg = _config(case)
        w = cfg.param_count()
        kv = B * cfg.num_layers * case["kv"] * cfg.num_kv_heads * cfg.head_dim
        att = 4 * B * cfg.num_layers * case["kv"] * cfg.num_q_heads * cfg.head_dim
        return {"bytes": 2 * (w + 2 * kv + B * (cfg.hidden + cfg.vocab)), "flops": 2 * B * w + att}
    if kind == "decode":
        # sequences of half to all of kv tokens, three quarters on average, one of kv
        tokens = case["kv"] * (1 + 0.75 * (B - 1))
        return {"bytes": 4 * tokens * case["hkv"] * 128 + 4 * B * case["hq"] * 128,
                "flops": 4 * tokens * case["hq"] * 128}
    if kind == "prefill":
        S, pairs = case["seq"], case["seq"] ** 2
        if case["causal"]:
            pairs = S * (S + 1) // 2
        return {"bytes": 4 * B * S * (case["hq"] + case["hkv"]) * 128, "flops": 4 * B * case["hq"] * 128 * pairs}
    if kind == "graph_attn":
        M, L, d = case["m"], case["kv"], case["d"]
        return {"bytes": 4 * B * (M + L) * d, "flops": 4 * B * M * L * d}
    K, N = case["k"], case["n"]
    mats = 2 if kind == "mlp" else 1
    io = B * K + B * N * (2 if case.get("residual") else 1) + (K if kind == "rms" else 0)
    more = 8 * B if kind == "head" else 0
    return {"bytes": 2 * (mats * K * N + io) + more, "flops": 2 * mats * B * K * N}


def tolerance(case):
    # single operators: fp32 sums, 16-bit tensors; another correct kernel may
    # round an intermediate 16-bit tensor (x * gamma, P, silu) elsewhere
    if case["kind"] == "step":
        return {"rel": 0.02, "max": 0.2, "differ": 0.01}
    rel = 0.01 if case.get("dtype") == "bf16" else 0.001  # about four times the error against 64 bits
    return {"rel": rel, "max": 10 * rel, "differ": 0.01}


# ------------------------------------------------------------------ 64 bits
def _rms(x):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + 1e-6)


def _exact_step(case, seed):
    cfg, B, L = _config(case), case["rows"], case["kv"]
    D, G, hkv = cfg.head_dim, cfg.num_q_heads // cfg.num_kv_heads, cfg.num_kv_heads
    ids, pages = _tokens_and_pages(case, seed)
    ids = torch.from_numpy(ids).cuda()
    pages = torch.from_numpy(pages).cuda().long().view(B, -1)
    inv = 1.0 / cfg.rope_theta ** (np.arange(0, D, 2, dtype=np.float64) / D)
    ang = torch.from_numpy(np.concatenate([inv, inv]) * (L - 1))
    cos, sin = ang.cos().to(torch.bfloat16).double().cuda(), ang.sin().to(torch.bfloat16).double().cuda()

    def rope(x):  # [B, heads, D] at position L - 1
        return x * cos + torch.cat([-x[..., D // 2:], x[..., : D // 2]], -1) * sin

    out = {"logits": None, "tokens": None, "k": [], "v": []}
    t, h = {}, None
    for layer, name, values in _checkpoint(case, seed):
        if name == "embed":
            h = values[ids].double()
        elif name == "norm":
            h = _rms(h) * values.double()
        elif name == "lm_head":
            out["logits"] = torch.cat([h @ w.double().t() for w in values.split(16384)], -1)
        else:
            t[name] = values.double()
        if name != "v":
            continue
        x = _rms(h) * t["ln1"]
        q = rope((x @ t["wq"].t()).view(B, -1, D))
        kc, vc = t["k"], t["v"]
        last, slot = pages[:, (L - 1) // 64], (L - 1) % 64
        kc[last, slot] = rope((x @ t["wk"].t()).view(B, hkv, D))
        vc[last, slot] = (x @ t["wv"].t()).view(B, hkv, D)
        att = torch.empty_like(q)
        for b in range(B):
            kb, vb = (c[pages[b]].reshape(-1, hkv, D)[:L] for c in (kc, vc))
            for g in range(hkv):
                p = torch.softmax(q[b, g * G:(g + 1) * G] @ kb[:, g].t() / math.sqrt(D), -1)
                att[b, g * G:(g + 1) * G] = p @ vb[:, g]
        h = h + att.view(B, -1) @ t["wo"].t()
        x = _rms(h) * t["ln2"]
        a, u = x @ t["wg"].t(), x @ t["wu"].t()
        h = h + (a * torch.sigmoid(a) * u) @ t["wd"].t()
        out["k"].append(kc.float())
        out["v"].append(vc.float())
        t = {}
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "step":
        return _exact_step(case, seed)
    if kind == "graph_attn":
        t = _graph_attn(case, seed)
        return [torch.stack([torch.softmax(q.double() @ k.double(), -1) @ v.double()
                             for q, k, v in zip(t["q"], t["k"], t["v"])])]
    if kind == "decode":
        t, G = _paged(case, seed), case["hq"] // case["hkv"]
        out = torch.empty(t["q"].shape, dtype=torch.float64, device="cuda")
        ptr, lens = t["indptr"].tolist(), t["lens"].tolist()
        for b in range(case["rows"]):
            pg = t["indices"][ptr[b]:ptr[b + 1]].long()
            kb, vb = (t[n][pg].reshape(-1, case["hkv"], 128)[: lens[b]].double() for n in ("k", "v"))
            for g in range(case["hkv"]):
                q = t["q"][b, g * G:(g + 1) * G].double()
                out[b, g * G:(g + 1) * G] = torch.softmax(q @ kb[:, g].t() / math.sqrt(128), -1) @ vb[:, g]
        return out
    if kind == "prefill":
        t, G, S = _prompt(case, seed), case["hq"] // case["hkv"], case["seq"]
        out = torch.empty(t["q"].shape, dtype=torch.float64, device="cuda")
        mask = torch.ones((S, S), dtype=torch.bool, device="cuda").triu(1) if case["causal"] else None
        for b in range(case["rows"]):
            for i in range(case["hq"]):
                a = t["q"][b, :, i].double() @ t["k"][b, :, i // G].double().t() / math.sqrt(128)
                if mask is not None:
                    a.masked_fill_(mask, -math.inf)
                out[b, :, i] = torch.softmax(a, -1) @ t["v"][b, :, i // G].double()
        return out
    t = _dense(case, seed)
    x = t["x"].double()
    if kind in ("rms", "graph_norm"):
        x = _rms(x) * (t["gamma"].double() if kind == "rms" else 1.0)
    kn = kind == "graph_norm" or case.get("layout", NK) == KN

    def product(w):  # in pieces of the output: the weight in 64 bits is large
        return torch.cat([x @ (p.double() if kn else p.double().t()) for p in w.split(8192, 1 if kn else 0)], -1)

    y = product(t["w"])
    if kind == "mlp":
        y = y * torch.sigmoid(y) * product(t["w3"])
    if "residual" in t:
        y = y + t["residual"].double()
    if kind == "head":
        return y, None
    return [y] if kind == "graph_norm" else y
