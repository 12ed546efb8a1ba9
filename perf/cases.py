"""Performance cases: what programs built on this framework have it do.

Each case is one call path through the public entry points (toyinfer_amd.attn,
toyinfer_amd.qwen3) at the geometries this repository is built for: Qwen3
attention heads (16/8 and 32/8, head_dim 128), head_dim 64, the 0.6B layer
(hidden 1024, MLP 3072, vocabulary 151936) and 4096-wide layers, prompts from a
few tokens to 8192, caches to 40960 rows.  Inputs are drawn on the GPU from a
seed; `exact` gives the same results in 64 bits with plain torch.
"""
import math

import torch

from toyinfer_amd import attn, qwen3

EPS, THETA = 1e-6, 1e6
VOCAB = 151936
# hidden, query heads, key/value heads, MLP width (head_dim 128)
WIDTHS = {1024: (16, 8, 3072), 4096: (32, 8, 12288)}


def listed():
    return [
        # The shortest prompt configuration: attention of one layer, launch-bound.
        {"name": "attention_s128", "kind": "attention", "s": 128, "hq": 16, "hkv": 8, "d": 128},
        # A chat prompt with its system text: attention of one 0.6B layer.
        {"name": "attention_s1371", "kind": "attention", "s": 1371, "hq": 16, "hkv": 8, "d": 128},
        # The smaller head size, a longer ragged prompt.
        {"name": "attention_s2985_d64", "kind": "attention", "s": 2985, "hq": 32, "hkv": 8,
         "d": 64},
        # A long document: QK-norm, RoPE and attention of one 32/8-head layer.
        {"name": "fused_s8192", "kind": "fused", "s": 8192, "hq": 32, "hkv": 8, "d": 128},
        # A serving step over eight sequences of different lengths.
        {"name": "decode_b8_l4096", "kind": "decode", "b": 8, "l": 4096, "hq": 32, "hkv": 8,
         "d": 128},
        # The drop-in decode call (probabilities and both outputs) deep in the
        # engine's 40960-row cache.
        {"name": "contract_pos32767", "kind": "contract", "pos": 32767, "msl": 40960, "hq": 32,
         "hkv": 8, "d": 128},
        # One decoder layer over a one-line prompt, and over the chat prompt.
        {"name": "layer_t37", "kind": "layer", "t": 37, "hidden": 1024},
        {"name": "layer_t1371", "kind": "layer", "t": 1371, "hidden": 1024},
        # One large prefill projection.
        {"name": "projection_t4096", "kind": "projection", "t": 4096, "m": 4096, "n": 4096},
        # Final norm and lm-head of a decode step.
        {"name": "head_h1024", "kind": "head", "vocab": VOCAB, "hidden": 1024},
        # The default sampler settings over one row of logits.
        {"name": "sample_k20", "kind": "sample", "vocab": VOCAB, "top_k": 20, "top_p": 0.95,
         "temperature": 0.6},
        # A whole request of the 0.6B model: prompt, then decode steps from the graph.
        {"name": "request_n1371", "kind": "request", "layers": 28, "n": 1371, "steps": 32},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["attention", "fused", "decode", "contract", "layer", "projection", "head",
                       "sample", "request"])
    hq, hkv = rng.choice([(16, 8), (32, 8), (8, 8), (12, 2), (6, 3)])
    d = rng.choice([128, 128, 64])
    if kind == "attention":
        return {"kind": kind, "s": _log_int(rng, 16, 4096), "hq": hq, "hkv": hkv, "d": d}
    if kind == "fused":
        return {"kind": kind, "s": _log_int(rng, 16, 8192), "hq": hq, "hkv": hkv, "d": d}
    if kind == "decode":
        b = _log_int(rng, 1, 32)
        return {"kind": kind, "b": b, "l": _log_int(rng, 32, 65536 // b), "hq": hq, "hkv": hkv,
                "d": d}
    if kind == "contract":
        pos = _log_int(rng, 8, 32768)
        return {"kind": kind, "pos": pos, "msl": rng.randint(pos + 1, 40960), "hq": hq,
                "hkv": hkv, "d": d}
    if kind == "layer":
        return {"kind": kind, "t": _log_int(rng, 5, 2048), "hidden": rng.choice(sorted(WIDTHS))}
    if kind == "projection":
        return {"kind": kind, "t": _log_int(rng, 1, 4096), "m": _log_int(rng, 256, 4096),
                "n": 64 * _log_int(rng, 8, 64)}
    if kind == "head":
        return {"kind": kind, "vocab": _log_int(rng, 8192, VOCAB), "hidden": 64 * rng.randint(8, 64)}
    if kind == "sample":
        return {"kind": kind, "vocab": _log_int(rng, 8192, VOCAB), "top_k": _log_int(rng, 2, 256),
                "top_p": round(rng.uniform(0.5, 0.99), 3),
                "temperature": round(rng.uniform(0.4, 1.3), 3)}
    return {"kind": kind, "layers": rng.randint(2, 28), "n": _log_int(rng, 5, 1371),
            "steps": rng.randint(1, 32)}


# ------------------------------------------------------------------ inputs

class _Rng:
    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(seed)

    def normal(self, *shape, std=1.0):
        return (torch.randn(shape, generator=self.g, device="cuda") * std).to(torch.bfloat16)

    def gamma(self, n):
        return (0.9 + 0.2 * torch.rand(n, generator=self.g, device="cuda")).to(torch.bfloat16)

    def ints(self, lo, hi, *shape):
        return torch.randint(lo, hi, shape, generator=self.g, device="cuda", dtype=torch.int32)


def _inputs(case, seed):
    """The tensors a case reads, by name, from the seed alone."""
    r, kind = _Rng(seed), case["kind"]
    if kind in ("attention", "fused"):
        s, hq, hkv, d = case["s"], case["hq"], case["hkv"], case["d"]
        t = {"q": r.normal(s, hq, d), "k": r.normal(s, hkv, d), "v": r.normal(s, hkv, d)}
        if kind == "fused":
            t["q_gamma"], t["k_gamma"] = r.gamma(d), r.gamma(d)
        return t
    if kind == "decode":
        b, l, hq, hkv, d = case["b"], case["l"], case["hq"], case["hkv"], case["d"]
        return {"q": r.normal(b, hq, d), "k": r.normal(b, l, hkv, d), "v": r.normal(b, l, hkv, d),
                "lens": r.ints((3 * l + 3) // 4, l + 1, b)}
    if kind == "contract":
        msl, hq, hkv, d = case["msl"], case["hq"], case["hkv"], case["d"]
        return {"q": r.normal(hq, d), "k": r.normal(msl, hkv, d), "v": r.normal(msl, hkv, d)}
    if kind == "layer":
        H = case["hidden"]
        return {"ids": r.ints(0, 4096, case["t"]), "embed": r.normal(4096, H),
                "w": _layer_weights(r, H, 1.0)}
    if kind == "projection":
        return {"x": r.normal(case["t"], case["n"]),
                "w": r.normal(case["m"], case["n"], std=case["n"] ** -0.5)}
    if kind == "head":
        H = case["hidden"]
        return {"x": r.normal(H), "gamma": r.gamma(H), "w": r.normal(case["vocab"], H, std=0.02)}
    if kind == "sample":
        return {"logits": torch.randn(case["vocab"], generator=r.g, device="cuda") * 2.5,
                "coin": torch.rand(1, generator=r.g, device="cuda")}
    # A trained model's next token stands well clear of the rest: the lm-head
    # rows are the embeddings moved along the vocabulary, and the residual
    # branches are small beside the embedding.
    L = case["layers"]
    embed = r.normal(VOCAB, 1024)
    shift = int(torch.randint(1, VOCAB, (1,), generator=r.g, device="cuda"))
    return {"ids": r.ints(0, VOCAB, case["n"]), "embed": embed,
            "head": (embed.float() * 0.02).to(torch.bfloat16).roll(shift, 0), "norm": r.gamma(1024),
            "layers": [_layer_weights(r, 1024, (2.0 * L) ** -0.5) for _ in range(L)]}


def _layer_weights(r, H, residual_scale):
    hq, hkv, F = WIDTHS[H]
    std = 0.02 * (1024 / H) ** 0.5
    out_std = std * residual_scale
    return {"input_layernorm": r.gamma(H), "q_proj": r.normal(hq * 128, H, std=std),
            "k_proj": r.normal(hkv * 128, H, std=std), "v_proj": r.normal(hkv * 128, H, std=std),
            "q_norm": r.gamma(128), "k_norm": r.gamma(128),
            "o_proj": r.normal(H, hq * 128, std=out_std),
            "post_attention_layernorm": r.gamma(H), "gate_proj": r.normal(F, H, std=std),
            "up_proj": r.normal(F, H, std=std), "down_proj": r.normal(H, F, std=out_std)}


def _bf16(*shape):
    return torch.empty(shape, dtype=torch.bfloat16, device="cuda")


def _rope_table(positions, d):
    inv = torch.empty(d // 2, device="cuda")
    table = torch.empty(positions, d // 2, 2, device="cuda")
    attn.precompute_freq_f32(inv, d, THETA)
    attn.rope_cos_sin_f32(table, inv, positions, d)
    return table


def prepare(case, seed):
    t, kind = _inputs(case, seed), case["kind"]
    st = {"case": case, **t}
    if kind in ("attention", "fused"):
        st["o"] = torch.empty_like(t["q"])
        if kind == "fused":
            st["k_out"] = torch.empty_like(t["k"])
            st["rope"] = _rope_table(case["s"], case["d"])
    elif kind == "decode":
        b, l, hq, hkv, d = case["b"], case["l"], case["hq"], case["hkv"], case["d"]
        st["splits"] = attn.decode_default_splits(b, hq, hkv, d, l)
        st["ws"] = attn.decode_workspace(b, hq, d, st["splits"], "cuda")
        st["o"] = torch.empty_like(t["q"])
    elif kind == "contract":
        hq, d = case["hq"], case["d"]
        st["pos_d"] = torch.tensor([case["pos"]], dtype=torch.int32, device="cuda")
        st["score"] = torch.empty(hq, case["msl"], device="cuda")
        st["o_buffer"] = torch.empty(hq, d, device="cuda")
        st["o"] = _bf16(hq, d)
    elif kind == "layer":
        T, H = case["t"], case["hidden"]
        hq, hkv, F = WIDTHS[H]
        st.update(hidden=_bf16(T, H), xn=_bf16(T, H), q=_bf16(T, hq * 128), k=_bf16(T, hkv * 128),
                  k_cache=_bf16(T, hkv * 128), v_cache=_bf16(T, hkv * 128), o=_bf16(T, hq * 128),
                  inter=_bf16(T, F), rope=_rope_table(T, 128))
    elif kind == "projection":
        st["y"] = _bf16(case["t"], case["m"])
    elif kind == "head":
        st["xn"] = torch.empty_like(t["x"])
        st["logits"] = torch.empty(case["vocab"], device="cuda")
    elif kind == "sample":
        st["token"] = torch.empty(1, dtype=torch.int32, device="cuda")
        st["ws"] = torch.zeros(attn.sample_workspace_bytes(), dtype=torch.uint8, device="cuda")
    else:
        hq, hkv, F = WIDTHS[1024]
        cfg = qwen3.make_config(num_layers=case["layers"], hidden_size=1024, num_q_heads=hq,
                                num_kv_heads=hkv, head_dim=128, intermediate_size=F,
                                vocab_size=VOCAB, max_seq_len=2048, max_prefill_tokens=1408,
                                rms_norm_eps=EPS, rope_theta=THETA)
        # The model works on a stream of its own: the weights come first.
        torch.cuda.synchronize()
        st["model"] = qwen3.Qwen3(cfg, {"embed_tokens": t["embed"], "norm": t["norm"],
                                        "lm_head": t["head"], "layers": t["layers"]})
    return st


# -------------------------------------------------------------------- runs

def run(st):
    c, kind = st["case"], st["case"]["kind"]
    if kind == "attention":
        attn.flash_attention_v1_bf16(st["q"], st["k"], st["v"], st["o"], c["hq"], c["hkv"], c["d"],
                                     c["s"])
        return st["o"]
    if kind == "fused":
        attn.prefill_qknorm_rope_attention_bf16(st["q"], st["k"], st["v"], st["o"], st["k_out"],
                                                st["q_gamma"], st["k_gamma"], st["rope"], EPS,
                                                c["hq"], c["hkv"], c["d"], c["s"])
        return st["o"], st["k_out"]
    if kind == "decode":
        attn.decode_attention_bf16(st["q"], st["k"], st["v"], st["o"], c["b"], c["hq"], c["hkv"],
                                   c["d"], st["lens"], c["l"], c["l"] * c["hkv"] * c["d"],
                                   st["splits"], st["ws"])
        return st["o"]
    if kind == "contract":
        attn.attention_bf16_graph(st["q"], st["k"], st["v"], st["score"], st["o_buffer"], st["o"],
                                  c["hq"], c["hkv"], c["d"], st["pos_d"], c["msl"])
        return st["score"], st["o_buffer"], st["o"]
    if kind == "layer":
        T, H, w = c["t"], c["hidden"], st["w"]
        hq, hkv, F = WIDTHS[H]
        qd, kv = hq * 128, hkv * 128
        attn.gather_embedding_bf16(st["embed"], st["ids"], st["hidden"], T, H, 4096)
        attn.batch_rmsnorm_bf16(st["hidden"], w["input_layernorm"], st["xn"], None, EPS, T, H)
        attn.gemm_segments_bf16(st["xn"], T, H, [w["q_proj"], w["k_proj"], w["v_proj"]],
                                [st["q"], st["k"], st["v_cache"]], [qd, kv, kv])
        attn.prefill_qknorm_rope_attention_bf16(st["q"], st["k"], st["v_cache"], st["o"],
                                                st["k_cache"], w["q_norm"], w["k_norm"],
                                                st["rope"], EPS, hq, hkv, 128, T)
        attn.gemm_segments_bf16(st["o"], T, qd, [w["o_proj"]], [st["hidden"]], [H], residual=True)
        attn.batch_rmsnorm_bf16(st["hidden"], w["post_attention_layernorm"], st["xn"], None, EPS,
                                T, H)
        attn.gemm_swiglu_bf16(st["xn"], T, H, w["gate_proj"], w["up_proj"], F, st["inter"])
        attn.gemm_segments_bf16(st["inter"], T, F, [w["down_proj"]], [st["hidden"]], [H],
                                residual=True)
        return st["hidden"], st["k_cache"], st["v_cache"]
    if kind == "projection":
        attn.batch_gemv_proj_bf16(st["w"], st["x"], st["y"], c["t"], c["m"], c["n"])
        return st["y"]
    if kind == "head":
        attn.rmsnorm_bf16(st["x"], st["gamma"], st["xn"], None, EPS, c["hidden"])
        attn.gemv_proj_bf162float(st["w"], st["xn"], st["logits"], c["vocab"], c["hidden"])
        return st["logits"]
    if kind == "sample":
        attn.sample_topk_topp_f32(st["logits"], c["vocab"], c["temperature"], c["top_k"],
                                  c["top_p"], st["coin"], st["token"], st["ws"])
        return st["token"]
    m, n = st["model"], c["n"]
    m.prefill(st["ids"], n)
    m.decode(c["steps"], True)
    return m.logits_host(), m.tokens_host(n + 1 + c["steps"])[n:]


# -------------------------------------------------------------------- work

def work(case):
    kind = case["kind"]
    if kind in ("attention", "fused"):
        s, hq, hkv, d = case["s"], case["hq"], case["hkv"], case["d"]
        b = 2 * s * d * (2 * hq + 2 * hkv)
        if kind == "fused":
            b += 2 * s * hkv * d + 4 * s * d
        return {"bytes": b, "flops": 2 * s * (s + 1) * hq * d}
    if kind == "decode":
        rows = case["b"] * case["l"] * 7 / 8
        return {"bytes": 4 * rows * case["hkv"] * case["d"] + 4 * case["b"] * case["hq"] * case["d"],
                "flops": 4 * rows * case["hq"] * case["d"]}
    if kind == "contract":
        L, hq, hkv, d = case["pos"] + 1, case["hq"], case["hkv"], case["d"]
        return {"bytes": 4 * L * hkv * d + 4 * hq * case["msl"] + 8 * hq * d,
                "flops": 4 * L * hq * d}
    if kind == "layer":
        T, H = case["t"], case["hidden"]
        hq, hkv, F = WIDTHS[H]
        params = H * 128 * (2 * hq + 2 * hkv) + 3 * H * F
        return {"bytes": 2 * params + 2 * T * (2 * H + 2 * hkv * 128),
                "flops": 2 * T * params + 2 * T * (T + 1) * hq * 128}
    if kind == "projection":
        t, m, n = case["t"], case["m"], case["n"]
        return {"bytes": 2 * (t * n + m * n + t * m), "flops": 2 * t * m * n}
    if kind == "head":
        v, h = case["vocab"], case["hidden"]
        return {"bytes": 2 * v * h + 4 * h + 4 * v, "flops": 2 * v * h}
    if kind == "sample":
        return {"bytes": 4 * case["vocab"] + 8, "flops": 2 * case["vocab"]}
    L, n, steps = case["layers"], case["n"], case["steps"]
    hq, hkv, F = WIDTHS[1024]
    params = L * (1024 * 128 * (2 * hq + 2 * hkv) + 3 * 1024 * F)
    head = VOCAB * 1024
    kv = 4 * L * hkv * 128
    return {"bytes": 2 * (params + head) * (1 + steps) + kv * (n + steps * (n + steps / 2)),
            "flops": 2 * params * (n + steps) + 2 * head * (1 + steps)
            + L * hq * 128 * (2 * n * (n + 1) + 4 * steps * n)}


# Four times the distance from the 64-bit values that was measured: bf16 results
# and probabilities (0.002), with bf16 tensors between the operations as well
# (0.003 to 0.0035), through a whole model (0.012).
REL = {"fused": 1.4e-2, "layer": 1.3e-2, "request": 4.8e-2}


def tolerance(case):
    return "exact" if case["kind"] == "sample" else {"rel": REL.get(case["kind"], 8e-3)}


# ------------------------------------------------------------ 64-bit values

def _rms(x, gamma):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * gamma


def _rope(x, first):
    """Rotate-half RoPE of x [S][heads][D] at positions first, first + 1, ..."""
    s, d = x.shape[0], x.shape[-1]
    i = torch.arange(d // 2, device=x.device, dtype=torch.float64)
    a = (first + torch.arange(s, device=x.device, dtype=torch.float64))[:, None] \
        * THETA ** (-2.0 * i / d)
    c, sn = a.cos()[:, None, :], a.sin()[:, None, :]
    lo, hi = x[..., :d // 2], x[..., d // 2:]
    return torch.cat([lo * c - hi * sn, hi * c + lo * sn], -1)


def _attend(q, k, v):
    """Causal attention of the last q.shape[0] positions of k, v, one head at a time."""
    s, hq, d = q.shape
    n, hkv = k.shape[0], k.shape[1]
    out = torch.empty_like(q)
    mask = torch.ones(s, n, dtype=torch.bool, device=q.device).triu(n - s + 1)
    for h in range(hq):
        p = (q[:, h] @ k[:, h * hkv // hq].T * d ** -0.5).masked_fill_(mask, -math.inf)
        out[:, h] = torch.softmax(p, -1) @ v[:, h * hkv // hq]
    return out


def _layer(x, w, past, first):
    """One decoder layer over x [S][H]; past holds the earlier K and V rows."""
    H = x.shape[1]
    hq, hkv, _ = WIDTHS[H]
    w = {n: a.double() for n, a in w.items()}
    h = _rms(x, w["input_layernorm"])
    q = _rope(_rms((h @ w["q_proj"].T).view(-1, hq, 128), w["q_norm"]), first)
    k = _rope(_rms((h @ w["k_proj"].T).view(-1, hkv, 128), w["k_norm"]), first)
    v = (h @ w["v_proj"].T).view(-1, hkv, 128)
    if past is not None:
        k, v = torch.cat([past[0], k]), torch.cat([past[1], v])
    x = x + _attend(q, k, v).reshape(-1, hq * 128) @ w["o_proj"].T
    h = _rms(x, w["post_attention_layernorm"])
    x = x + (torch.nn.functional.silu(h @ w["gate_proj"].T) * (h @ w["up_proj"].T)) \
        @ w["down_proj"].T
    return x, (k, v)


def exact(case, seed):
    t, kind = _inputs(case, seed), case["kind"]
    if kind == "attention":
        return _attend(t["q"].double(), t["k"].double(), t["v"].double())
    if kind == "fused":
        q = _rope(_rms(t["q"].double(), t["q_gamma"].double()), 0)
        k = _rope(_rms(t["k"].double(), t["k_gamma"].double()), 0)
        return _attend(q, k, t["v"].double()), k
    if kind == "decode":
        return torch.cat([_attend(t["q"][b:b + 1].double(), t["k"][b, :n].double(),
                                  t["v"][b, :n].double())
                          for b, n in enumerate(t["lens"].tolist())])
    if kind == "contract":
        L, hq, hkv, d = case["pos"] + 1, case["hq"], case["hkv"], case["d"]
        q, k, v = t["q"].double(), t["k"][:L].double(), t["v"][:L].double()
        score = torch.zeros(hq, case["msl"], dtype=torch.float64, device="cuda")
        o = torch.empty(hq, d, dtype=torch.float64, device="cuda")
        for h in range(hq):
            score[h, :L] = torch.softmax(k[:, h * hkv // hq] @ q[h] * d ** -0.5, -1)
            o[h] = score[h, :L] @ v[:, h * hkv // hq]
        return score, o, o
    if kind == "layer":
        x, (k, v) = _layer(t["embed"][t["ids"].long()].double(), t["w"], None, 0)
        return x, k.reshape(case["t"], -1), v.reshape(case["t"], -1)
    if kind == "projection":
        return t["x"].double() @ t["w"].double().T
    if kind == "head":
        return t["w"].double() @ _rms(t["x"].double(), t["gamma"].double())
    if kind == "sample":
        x, at = (t["logits"].double() / case["temperature"]).topk(min(case["top_k"], case["vocab"]))
        p = torch.softmax(x / case["temperature"], -1)
        run_sum = p.cumsum(-1)
        over = (run_sum > case["top_p"]).nonzero()
        kept = int(over[0]) + 1 if len(over) else len(p)
        r = t["coin"].double() * run_sum[kept - 1]
        pick = (run_sum[:kept] > r).nonzero()
        return at[int(pick[0]) if len(pick) else kept - 1].to(torch.int32).reshape(1)
    embed, head = t["embed"], t["head"].double()
    ids, past, tokens, first = t["ids"].long(), [None] * case["layers"], [], 0
    for _ in range(case["steps"] + 1):
        x = embed[ids].double()
        for l, w in enumerate(t["layers"]):
            x, past[l] = _layer(x, w, past[l], first)
        first += len(ids)
        logits = head @ _rms(x[-1], t["norm"].double())
        ids = logits.argmax().reshape(1)
        tokens.append(int(ids))
    return logits, torch.tensor(tokens, dtype=torch.int64, device="cuda")
