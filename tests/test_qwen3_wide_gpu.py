"""The model harness at Qwen3-8B's layer widths (hidden 4096, 32/8 heads,
D=128, SwiGLU 12288; one layer, vocab 4096, tied embeddings; bf16 weights
0.02 * N(0, 1), norm weights 1): a 24-token prefill and 3 greedy decode
steps, direct and from a captured graph, against the oracle's forward.

These widths take the decode projections down paths the 0.6B geometry does
not: inputs of 4096 elements (eight 16-byte chunks per lane in the one-token
GEMV, its largest register form) and the 12288-element input of the down
projection (the block-cooperative GEMV, for inputs over 4096).

Bars as for configuration 5 (tests/test_qwen3_config5_gpu.py): the oracle
and the device round the same activations to bf16 at the same points, and
their fp32 reduction orders differ.
"""
import numpy as np
import pytest
import torch

import oracle
from tests import helpers as H
from tests import qwen3_weights as QW
from toyinfer_amd import qwen3

pytestmark = pytest.mark.gpu

LOGIT_MAX_ABS = 0.1
LOGIT_MEAN_ABS = 0.02

WIDE = dict(num_layers=1, hidden_size=4096, num_q_heads=32, num_kv_heads=8, head_dim=128,
            intermediate_size=12288, vocab_size=4096, max_seq_len=64, max_prefill_tokens=32,
            rms_norm_eps=1e-6, rope_theta=1e6)
SEED = 93


@pytest.fixture(scope="module")
def weights_wide(dev):
    print("[step] wide weights (host draw + upload)", flush=True)
    bits = QW.weight_bits(WIDE, SEED, proj_std=0.02, embed_std=0.02, norm_range=None, tied=True)
    dw = {"layers": [{n: H.to_dev_bf16(b, dev) for n, b in lw.items()} for lw in bits["layers"]]}
    dw["embed_tokens"] = H.to_dev_bf16(bits["embed_tokens"], dev)
    dw["norm"] = H.to_dev_bf16(bits["norm"], dev)
    dw["lm_head"] = dw["embed_tokens"]
    host = QW.to_f32(bits)
    host["inv_freq"] = oracle.inv_freq(WIDE["head_dim"], WIDE["rope_theta"])
    H.sync()
    return host, dw


def check_logits(got, exp, label):
    assert np.isfinite(got).all(), f"{label}: non-finite logits"
    d = np.abs(got.astype(np.float64) - exp)
    print(f"  {label}: max {d.max():.4f} mean {d.mean():.5f} (std {exp.std():.3f})", flush=True)
    assert d.max() <= LOGIT_MAX_ABS and d.mean() <= LOGIT_MEAN_ABS, \
        f"{label}: max {d.max():.3g} mean {d.mean():.3g}"


# max_seq_len 64: the attention pass gives each split a fixed 128-row slice of
# the cache and requests it before the device length arrives; 16384 (more
# rows than 96 splits x 128): slices follow the length instead.
@pytest.mark.parametrize("msl", [64, 16384])
@pytest.mark.parametrize("graph", [False, True])
def test_wide_prefill_and_decode_vs_oracle(dev, weights_wide, graph, msl):
    print(f"[step] wide prefill 24 + 3 decode steps, graph={graph}, max_seq_len={msl}", flush=True)
    host, dw = weights_wide
    T, steps = 24, 3
    ids = np.random.default_rng(SEED + int(graph)).integers(0, WIDE["vocab_size"], T)
    ids = ids.astype(np.uint32)
    m = qwen3.Qwen3(qwen3.Config(**dict(WIDE, max_seq_len=msl)), dw)
    id_t = torch.from_numpy(ids.view(np.int32)).to(dev)
    m.prefill(id_t, T)
    got = m.logits_host()
    ref = oracle.Qwen3Reference(dict(WIDE, max_seq_len=T + steps + 1), host)
    check_logits(got, ref.forward(ids, 0), "prefill")
    toks = m.tokens_host(T + 1)
    assert toks[T] == oracle.argmax(got), "prefill pick"
    for s in range(steps):
        m.decode(1, graph)
        got = m.logits_host()
        toks = m.tokens_host(T + s + 2)
        check_logits(got, ref.forward([toks[T + s]], T + s), f"step {s}")
        assert toks[T + s + 1] == oracle.argmax(got), f"step {s} pick"
    assert m.position_host() == T + steps
    m.close()


# One-token projections with the norm in front: the input requested ahead of
# the weight rows or in trips with them, by grid size and row length (n = 1536,
# 2560, 3584 and 4096 on either side of the lines: q/k/v of 1024, 4608, 6144 and
# 8192 rows, gate/up of 1024 to 4096).
@pytest.mark.parametrize("hidden,hq,hkv,F", [(1536, 4, 2, 1536), (1536, 32, 8, 4096),
                                             (2560, 8, 4, 2048), (2560, 32, 16, 2560),
                                             (3584, 28, 4, 1024), (4096, 8, 4, 1024)])
def test_decode_projection_orders_vs_prefill(dev, hidden, hq, hkv, F):
    """The logits of a decode step equal, within the oracle bars, those of a
    prefill that ends with the same token (whose projections are GEMMs)."""
    print(f"[step] decode projections hidden={hidden} {hq}/{hkv} F={F}", flush=True)
    g = torch.Generator(device=dev).manual_seed(SEED)
    V, T = 512, 24

    def draw(*shape):
        return (torch.randn(shape, generator=g, device=dev) * 0.02).to(torch.bfloat16)

    ones = torch.ones(hidden, dtype=torch.bfloat16, device=dev)
    layer = {"input_layernorm": ones, "q_proj": draw(hq * 128, hidden),
             "k_proj": draw(hkv * 128, hidden), "v_proj": draw(hkv * 128, hidden),
             "q_norm": ones[:128], "k_norm": ones[:128], "o_proj": draw(hidden, hq * 128),
             "post_attention_layernorm": ones, "gate_proj": draw(F, hidden),
             "up_proj": draw(F, hidden), "down_proj": draw(hidden, F)}
    embed = draw(V, hidden)
    ids = torch.randint(0, V, (T + 1,), generator=g, device=dev, dtype=torch.int32)
    H.sync()
    cfg = qwen3.make_config(num_layers=1, hidden_size=hidden, num_q_heads=hq, num_kv_heads=hkv,
                            head_dim=128, intermediate_size=F, vocab_size=V, max_seq_len=64,
                            max_prefill_tokens=32, rms_norm_eps=1e-6, rope_theta=1e6)
    m = qwen3.Qwen3(cfg, {"embed_tokens": embed, "norm": ones, "lm_head": embed, "layers": [layer]})
    m.prefill(ids, T)
    pick = int(m.tokens_host(T + 1)[T])
    m.decode(1, True)
    got = m.logits_host()
    ids[T] = pick
    H.sync()
    m.prefill(ids, T + 1)
    check_logits(got, m.logits_host(), "decode vs prefill")
    m.close()
