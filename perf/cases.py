"""The work that a user of this package has it do, as measurable cases.

One case is one pass through public entry points: a decode-attention step over a hybrid cache, a quantise-and-append,
the reconstruction of a dense cache, the attention of a prompt, a compression, or a short generation of one attention
layer of either kind.  Shapes are those of the package's own configurations (``hqekv_amd.synth.CONFIGS``, the benchmark)
and of the models that run on it: 32 query and 8 KV heads of 128 channels, and the other group sizes it supports.
Data is synthetic: K and V ~ N(0, 1) with four outlier channels of K scaled by ten, q ~ N(0, 1)."""
from __future__ import annotations

import math

import torch

from hqekv_amd import synth
from hqekv_amd.attention import DecodePlan
from hqekv_amd.decode_layer import (HqeAttentionLayer, class_token_counts, gqa_prompt_attention, last_rows_probabilities,
                                    ratios_for_next_increment)
from hqekv_amd.hqe_2 import KV_cache_hqe_2, KV_cache_reconstruct_hqe
from hqekv_amd.hqe_matmul import qkv_matmul_hqe_2
from hqekv_amd.kivi_layer import KiviAttentionLayer
from hqekv_amd.pack_unpack import quantize_pack_into, uniform_group_quantize_pack_last_dim
from hqekv_amd.public_func import last_attn_weights

D = 128
LAST_ROWS = 20
HEADS = ((32, 8), (40, 8), (24, 8), (28, 4))   # query and KV heads: groups of 4, 5, 3 and 7
BITS = (16, 8, 4, 2, 1)
# shares of fp16, 8, 4, 2 bit and evicted tokens of the package's four decode configurations
MIXES = {name: cfg["fractions"] for name, cfg in synth.CONFIGS.items()}
# evicted, 4, 2 and 1 bit shares of the layers: without the 1-bit class, and with the normal-quantile one
RATIOS = {"uniform_group": (0.20, 0.48, 0.32, 0.0),
          "high_uniform_group_low_normal_group": (0.20, 0.25, 0.30, 0.25)}
LOW_NORMAL = "high_uniform_group_low_normal_group"


def listed():
    return [
        # the first tokens after a short chat prompt: latency, launches and host work are everything
        dict(name="decode_1k", kind="decode", entry="call", B=1, Hq=32, Hkv=8, T=1056, residual=17, mix="c2"),
        # the headline configuration, one 32k-token conversation, from a serving loop that keeps its plan
        dict(name="decode_32k", kind="decode", entry="plan", B=1, Hq=32, Hkv=8, T=32768, residual=0, mix="c2"),
        # a small batch on a model with five query heads per KV head, a ragged residual in flight
        dict(name="decode_16k_b3_group5", kind="decode", entry="call", B=3, Hq=40, Hkv=8, T=16416, residual=29, mix="c5"),
        # batched long-context serving
        dict(name="decode_65k_b8", kind="decode", entry="plan", B=8, Hq=32, Hkv=8, T=65536, residual=0, mix="c4"),
        # 8k new tokens appended to a cache of 24k
        dict(name="quantize_8k_2bit", kind="quantize", B=1, Hkv=8, tokens=8192, at=24576, bits=2),
        # the prompts of a batch quantised into a new cache
        dict(name="quantize_64k_b4_4bit", kind="quantize", B=4, Hkv=8, tokens=65536, at=0, bits=4),
        # a cache turned back into dense K and V (handing a sequence over, checking accuracy)
        dict(name="reconstruct_16k", kind="reconstruct", B=1, Hkv=8, T=16384, residual=23, mix="c2"),
        # a short prompt of no round length, slices of a fused projection
        dict(name="prompt_1k", kind="prompt", B=1, Hq=32, Hkv=8, T=1003, fused=True),
        # a long prompt
        dict(name="prompt_32k", kind="prompt", B=1, Hq=32, Hkv=8, T=32768, fused=False),
        # what happens in a layer every 32 tokens of a long generation
        dict(name="compress_32k", kind="compress", B=1, T=32768, strategy="uniform_group"),
        # one layer of a short answer: prompt, its compression, decode steps
        dict(name="generate_4k", kind="generate", B=1, T=4099, steps=24, strategy=LOW_NORMAL),
        # the same for the layer that keeps every token; a block of keys is quantised on the way
        dict(name="kivi_generate_4k", kind="kivi", B=1, T=4080, steps=24, bits=2),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("decode",) * 5 + ("quantize",) * 2 + ("reconstruct",) + ("prompt",) * 2 + ("compress",) + ("generate",) + ("kivi",))
    if kind == "decode":
        Hq, Hkv = rng.choice(HEADS[:1] * 5 + HEADS[1:])
        T = max(16, _log(rng, 512, 131072) // 32) * 32
        B = min(rng.choice((1, 1, 2, 3, 4, 8, 16)), max(1, 8 * 65536 // T))
        return dict(kind=kind, entry=rng.choice(("call", "plan")), B=B, Hq=Hq, Hkv=Hkv, T=T,
                    residual=rng.choice((0, rng.randrange(1, 64))), mix=rng.choice(sorted(MIXES)))
    if kind == "quantize":
        tokens = max(1, _log(rng, 32, 65536) // 32) * 32
        return dict(kind=kind, B=min(rng.choice((1, 2, 4, 8)), max(1, 4 * 65536 // tokens)), Hkv=rng.choice((4, 8, 8)),
                    tokens=tokens, at=32 * rng.randrange(0, 1024), bits=rng.choice((1, 2, 2, 4, 4, 8)))
    if kind == "reconstruct":
        T = max(16, _log(rng, 512, 65536) // 32) * 32
        return dict(kind=kind, B=min(rng.choice((1, 2, 4)), max(1, 131072 // T)), Hkv=8, T=T,
                    residual=rng.choice((0, rng.randrange(1, 64))), mix=rng.choice(sorted(MIXES)))
    if kind == "prompt":
        Hq, Hkv = rng.choice(HEADS[:1] * 5 + HEADS[1:])
        T = _log(rng, 64, 32768 * 32 // Hq)
        B = min(rng.choice((1, 1, 2, 4)), max(1, 32 * 32768 ** 2 // (Hq * T * T)))
        return dict(kind=kind, B=B, Hq=Hq, Hkv=Hkv, T=T, fused=rng.choice((True, False)))
    if kind == "compress":
        T = _log(rng, 1024, 131072) // 32 * 32
        return dict(kind=kind, B=min(rng.choice((1, 2, 4)), max(1, 262144 // T)), T=T, strategy=rng.choice(sorted(RATIOS)))
    if kind == "generate":
        T = max(8, _log(rng, 256, 8192) // 32) * 32 + rng.randrange(0, 8)   # the steps end before the next compression
        return dict(kind=kind, B=rng.choice((1, 2)), T=T, steps=rng.randrange(8, 25 - T % 32), strategy=rng.choice(sorted(RATIOS)))
    return dict(kind=kind, B=rng.choice((1, 2)), T=_log(rng, 200, 8192), steps=rng.randrange(8, 25), bits=rng.choice((2, 2, 4)))


# ---------------------------------------------------------------------------------------------------- inputs
def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _normal(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float16)


def _keys(g, *shape):
    k = _normal(g, *shape)
    for c in synth.OUTLIER_CHANNELS:
        k[..., c] *= 10.0
    return k


def _hybrid_cache(case, g, seed):
    T = case["T"] + case["residual"]
    k, v = _keys(g, case["B"], case["Hkv"], T, D), _normal(g, case["B"], case["Hkv"], T, D)
    classes = synth.split_blocks(case["T"], MIXES[case["mix"]], seed)
    return synth.build_cache(k, v, classes, case["residual"], uniform_group_quantize_pack_last_dim)


def prepare(case, seed):
    g = _generator(seed)
    kind, B = case["kind"], case["B"]
    if kind == "decode":
        pkv = _hybrid_cache(case, g, seed)
        q = _normal(g, B, case["Hq"], 1, D)
        return dict(case=case, q=q, pkv=pkv, plan=DecodePlan(q, pkv) if case["entry"] == "plan" else None)
    if kind == "quantize":
        n, at, bits, H = case["tokens"], case["at"], case["bits"], case["Hkv"]
        pf, cap = 32 // bits, case["at"] + case["tokens"]
        i32, f16 = dict(dtype=torch.int32, device="cuda"), dict(dtype=torch.float16, device="cuda")
        kc, vc = torch.zeros(B, H, D, cap // pf, **i32), torch.zeros(B, H, cap, D // pf, **i32)
        ks, kz = torch.zeros(B, H, D, cap // 32, **f16), torch.zeros(B, H, D, cap // 32, **f16)
        vs, vz = torch.zeros(B, H, cap, D // 32, **f16), torch.zeros(B, H, cap, D // 32, **f16)
        return dict(case=case, k=_keys(g, B, H, n, D), v=_normal(g, B, H, n, D),
                    k_out=(kc[..., at // pf:], ks[..., at // 32:], kz[..., at // 32:]),
                    v_out=(vc[:, :, at:], vs[:, :, at:], vz[:, :, at:]))
    if kind == "reconstruct":
        return dict(case=case, pkv=_hybrid_cache(case, g, seed))
    if kind == "prompt":
        Hq, Hkv, T = case["Hq"], case["Hkv"], case["T"]
        if case["fused"]:   # what a fused projection hands over: (B, T, heads, D), seen per head
            y = _normal(g, B, T, Hq + 2 * Hkv, D).transpose(1, 2)
            q, k, v = y[:, :Hq], y[:, Hq:Hq + Hkv], y[:, Hq + Hkv:]
        else:
            q, k, v = _normal(g, B, Hq, T, D), _normal(g, B, Hkv, T, D), _normal(g, B, Hkv, T, D)
        return dict(case=case, q=q, k=k, v=v)
    if kind == "compress":
        # A prompt compressed as a layer does it, 32 tokens decoded since.  Nothing was evicted, as in nearly every later
        # compression of a long generation, and the newest tokens hold the most attention: so the classes of all seeds
        # have the same sizes.
        T, strategy = case["T"], case["strategy"]
        ring = last_attn_weights(last_length=LAST_ROWS)
        ring.set_max_length(T + 64)
        # recent rows of probabilities, summed over batch and heads: a few tokens hold most of the mass, in every row
        rows = torch.exp(2.0 * torch.randn(T, generator=g, device="cuda") + 0.3 * torch.randn(1, 1, LAST_ROWS, T, generator=g, device="cuda"))
        rows[..., T - 32:] = 400 * rows.mean()
        ring.update((rows * (32.0 * B) / rows.sum(-1, keepdim=True)).half())
        importance, order = ring.ranked_importance(T)
        shares = torch.tensor(RATIOS[strategy][1:])
        ratio_e, ratio_q = torch.zeros(1), shares / shares.sum()
        n = class_token_counts(T, ratio_q, ratio_e)[1]
        pkv = (None,) * 39 + (_keys(g, B, 8, T, D), _normal(g, B, 8, T, D), T)
        pkv = KV_cache_hqe_2(pkv, T, 0, order, n, n.clone(), importance, strategy, ring)
        row = ring.weights[:1, :T + 32].clone()   # the last step looked at the old tokens as before
        row[:, T:] = row[:, T - 32:T]
        ring.update(row.view(1, 1, 1, T + 32))
        pkv = pkv[:39] + (_keys(g, B, 8, 32, D), _normal(g, B, 8, 32, D), T + 32)
        ratio_e, ratio_q = ratios_for_next_increment(T, ratio_e, ratio_q)
        return dict(case=case, pkv=pkv, ring=ring, counts=class_token_counts(T + 32, ratio_q, ratio_e)[1])
    T, S = case["T"], case["steps"]
    prompt = (_normal(g, B, 32, T, D), _keys(g, B, 8, T, D), _normal(g, B, 8, T, D))
    steps = [(_normal(g, B, 32, 1, D), _keys(g, B, 8, 1, D), _normal(g, B, 8, 1, D)) for _ in range(S)]
    if kind == "generate":
        evict, b4, b2, b1 = RATIOS[case["strategy"]]
        layer = HqeAttentionLayer(D, bit_0=evict, bit_4=b4, bit_2=b2, bit_1=b1, quant_strategy=case["strategy"])
    else:
        layer = KiviAttentionLayer(D, k_bits=case["bits"], v_bits=case["bits"])
    return dict(case=case, layer=layer, prompt=prompt, steps=steps)


# ---------------------------------------------------------------------------------------------------- one pass
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "decode":
        if state["plan"] is not None:
            return state["plan"].run(state["q"])
        return qkv_matmul_hqe_2(state["q"], state["pkv"], None, D, "uniform_group")
    if kind == "quantize":
        quantize_pack_into(state["k"].transpose(2, 3), case["bits"], *state["k_out"])
        quantize_pack_into(state["v"], case["bits"], *state["v_out"])
        return state["k_out"], state["v_out"]
    if kind == "reconstruct":
        return KV_cache_reconstruct_hqe(state["pkv"], "uniform_group")
    if kind == "prompt":
        q, k, v = state["q"], state["k"], state["v"]
        scaling = D ** -0.5
        return last_rows_probabilities(q, k, None, scaling, LAST_ROWS), gqa_prompt_attention(q, k, v, None, scaling)
    if kind == "compress":
        ring, n = state["ring"], state["counts"]
        importance, order = ring.ranked_importance(case["T"] + 32)
        pkv = KV_cache_hqe_2(state["pkv"], 32, case["T"], order, n, n.clone(), importance, case["strategy"], ring)
        return pkv, ring.weights
    layer, outs = state["layer"], []
    if kind == "generate":
        layer.reset()
        layer.set_max_length(case["T"] + case["steps"])
        out, weights, pkv, _ = layer(*state["prompt"])
        for q, k, v in state["steps"]:
            outs.append(out)
            out, weights, pkv, _ = layer(q, k, v, None, pkv)
        return outs, out, weights, layer.last_weights.weights, pkv
    out, weights, pkv = layer(*state["prompt"])
    for q, k, v in state["steps"]:
        outs.append(out)
        out, weights, pkv = layer(q, k, v, None, pkv)
    return outs, out, weights, pkv


# ---------------------------------------------------------------------------------------------------- what it takes
def _side_bytes(B, Hkv, tokens_by_bits):
    """One side of a cache: codes, scale and zero (or fp16 rows) of every KV head, and a position per token."""
    return sum(n * (B * Hkv * (2 * D if b == 16 else D * b // 8 + D // 32 * 4) + 8) for b, n in tokens_by_bits.items())


def _mix_tokens(case):
    counts = synth.block_counts(case["T"] // 32, MIXES[case["mix"]])
    return {b: 32 * c for b, c in zip(synth.CLASS_ORDER, counts) if b}


def _layer_tokens(n, strategy, evicted=True):
    shares = torch.tensor(RATIOS[strategy])
    if not evicted:
        shares[0] = 0.0
    return {b: int(c) for b, c in zip(BITS, class_token_counts(n, shares[1:] / shares[1:].sum() * (1 - shares[0]), shares[:1])[1])}


def work(case):
    kind, B = case["kind"], case["B"]
    if kind == "decode":
        tokens, Hq, Hkv = _mix_tokens(case), case["Hq"], case["Hkv"]
        n = sum(tokens.values()) + case["residual"]
        side = _side_bytes(B, Hkv, tokens) + B * Hkv * case["residual"] * 2 * D
        return dict(bytes=2 * side + B * Hq * (4 * D + 2 * n), flops=4 * B * Hq * n * D)
    if kind == "quantize":
        elems = 2 * B * case["Hkv"] * case["tokens"] * D
        return dict(bytes=elems * 2 + elems * case["bits"] // 8 + elems // 32 * 4, flops=4 * elems)
    if kind == "reconstruct":
        tokens = _mix_tokens(case)
        n = sum(tokens.values()) + case["residual"]
        dense = 2 * B * case["Hkv"] * D * 2
        return dict(bytes=2 * _side_bytes(B, case["Hkv"], tokens) + dense * (case["residual"] + n), flops=2 * B * case["Hkv"] * D * n * 2)
    if kind == "compress":
        side = _side_bytes(B, 8, _layer_tokens(case["T"], case["strategy"], evicted=False))
        return dict(bytes=2 * (2 * side + B * 8 * 32 * 2 * D) + LAST_ROWS * 2 * 2 * case["T"], flops=LAST_ROWS * case["T"])
    Hq, Hkv, T = case.get("Hq", 32), case.get("Hkv", 8), case["T"]
    rows = T * (T + 1) // 2
    bytes_, flops = B * T * D * 2 * (2 * Hq + 2 * Hkv), 4 * B * Hq * D * rows
    if kind in ("prompt", "generate"):
        bytes_ += B * Hq * LAST_ROWS * T * 2
        flops += 2 * B * Hq * D * LAST_ROWS * T
    if kind == "prompt":
        return dict(bytes=bytes_, flops=flops)
    tokens = _layer_tokens(T // 32 * 32, case["strategy"]) if kind == "generate" else {case["bits"]: max(0, T - 128), 16: min(T, 128)}
    side, n = _side_bytes(B, 8, tokens), sum(tokens.values())
    return dict(bytes=bytes_ + 2 * side + case["steps"] * (2 * side + B * 32 * (4 * D + 2 * n)),
                flops=flops + case["steps"] * 4 * B * 32 * n * D)


def tolerance(case):
    if case["kind"] in ("quantize", "reconstruct", "compress"):
        return "exact"   # codes, scales, zeros, positions and the values they stand for are defined to the bit
    # Scores are rounded to fp16 before the softmax, and so are probabilities and outputs: a score whose fp32 sum sits
    # next to the middle between two fp16 numbers moves by one place with the order of the additions, its probability by
    # half a percent.  Codes, scales and positions in the outputs stay the same.
    return {"rel": 3e-3, "max": 5e-2}
