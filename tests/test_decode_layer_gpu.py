"""The decode caller (prompt -> cache tuple -> decode steps with periodic compression) on the HIP path
against the oracle's restatement of the same layer, in lockstep.

The oracle's ring is fed with the probabilities the GPU produced (and, after each call, aligned to the
GPU ring bit for bit), so both sides take their policy decisions from identical importance values and the
caches can be compared bit for bit after every call; the probabilities and outputs themselves are compared
with the attention tolerance (1e-3 relative + 2e-3 absolute)."""
import pytest
import torch

from oracle import hqe_oracle as O

pytestmark = pytest.mark.gpu

RTOL, ATOL = 1e-3, 2e-3


def _qkv(B, Hq, Hkv, L, D, seed):
    g = torch.Generator().manual_seed(seed)
    q = torch.randn(B, Hq, L, D, generator=g)
    k = torch.randn(B, Hkv, L, D, generator=g)
    for ch in (3, 35, 67, 99):
        k[..., ch] *= 10.0
    v = torch.randn(B, Hkv, L, D, generator=g)
    return q.half(), k.half(), v.half()


def _causal_mask(T):
    m = torch.full((T, T), torch.finfo(torch.float16).min, dtype=torch.float16)
    return torch.triu(m, diagonal=1)[None, None]


def _same_tuple(got, want, where, normal=False):
    assert len(got) == len(want) == 42
    for i, (a, b) in enumerate(zip(got, want)):
        if i == 41:
            assert int(a) == int(b), (where, i)
            continue
        assert (a is None) == (b is None), (where, i)
        if a is None:
            continue
        a = a.cpu()
        assert a.shape == b.shape and a.dtype == b.dtype, (where, i, a.shape, b.shape)
        if a.dtype == torch.float16:
            assert torch.equal(a.view(torch.int16), b.view(torch.int16)), (where, i)
        else:
            assert torch.equal(a, b), (where, i)


@pytest.mark.parametrize("B,Hq,Hkv,T0,steps,strategy,bit_1", [
    (1, 8, 2, 300, 72, "uniform_group", 0.0),
    (2, 4, 4, 96, 40, "uniform_group", 0.0),
    (1, 8, 2, 300, 72, "high_uniform_group_low_normal_group", 0.25),   # the reference's shipped default
    (1, 4, 2, 20, 70, "uniform_group", 0.0),                            # prompt shorter than one block
    (2, 16, 4, 511, 40, "high_uniform_group_low_normal_group", 0.1),    # ragged prompt, GQA 4, two batch rows
    (1, 6, 2, 200, 40, "uniform_group", 0.0),                           # three query heads per KV head
    (2, 12, 2, 130, 40, "high_uniform_group_low_normal_group", 0.1),    # six per KV head
])
def test_layer_in_lockstep_with_oracle(dev, B, Hq, Hkv, T0, steps, strategy, bit_1):
    from hqekv_amd.decode_layer import HqeAttentionLayer
    D = 128
    ratios = dict(bit_0=0.2, bit_4=0.3, bit_2=0.5 - bit_1, bit_1=bit_1)
    layer = HqeAttentionLayer(D, **ratios, quant_strategy=strategy)
    layer.set_max_length(T0 + steps)
    orc = O.DecodeLayerOracle(D, **ratios, max_length=T0 + steps, quant_strategy=strategy)

    pkv_g = pkv_o = None
    compressions = 0
    for step in range(steps + 1):
        L = T0 if step == 0 else 1
        q, k, v = _qkv(B, Hq, Hkv, L, D, 4200 + step)
        mask = _causal_mask(T0) if step == 0 else None
        out_g, w_g, pkv_g, aux_g = layer(q.to(dev), k.to(dev), v.to(dev),
                                         None if mask is None else mask.to(dev), pkv_g, None)
        w_obs = w_g.cpu()
        out_o, w_o, pkv_o, aux_o = orc.step(q, k, v, mask, pkv_o, None,
                                            observed=w_obs if step else None)
        if step == 0:   # the oracle keeps every prompt row, the layer the last 20
            w_o = w_o[:, :, -w_obs.shape[2]:, :]
        where = f"step {step}"
        assert torch.allclose(w_obs.float(), w_o.float(), rtol=RTOL, atol=ATOL), where
        # the prompt's output comes from torch's fused attention (outside the quantised path): looser there
        o_rtol, o_atol = (RTOL, ATOL) if step else (1e-2, 1e-2)
        assert torch.allclose(out_g.cpu().float(), out_o.float(), rtol=o_rtol, atol=o_atol), where
        assert (aux_g is None) == (aux_o is None), where
        if aux_g is not None:
            compressions += 1
            assert torch.equal(aux_g[1], aux_o[1]) and torch.equal(aux_g[2], aux_o[2]), where
        assert layer.current_length == orc.current_length, where
        assert layer.history_reserve_length == orc.history_reserve_length, where
        assert torch.equal(layer.ratio_e, orc.ratio_e) and torch.equal(layer.ratio_q, orc.ratio_q), where
        # rings: the same rows summed on the GPU and on the CPU, then aligned exactly
        ring_g = layer.last_weights.weights.cpu()
        assert torch.allclose(ring_g.float(), orc.ring.weights.float(), rtol=2e-3, atol=1e-3), where
        assert layer.last_weights.next_line == orc.ring.next_line, where
        orc.ring.weights.copy_(ring_g)
        _same_tuple(pkv_g, pkv_o, where, normal=strategy != "uniform_group")
    assert compressions >= 2
    kept = sum(pkv_g[s].shape[2] for s in (2, 8, 16, 24, 32) if pkv_g[s] is not None)
    assert kept == layer.history_reserve_length
    assert int(pkv_g[41]) == T0 + steps


@pytest.mark.parametrize("fused", [True, False], ids=["one-call", "separate"])
def test_layer_tuples_keep_their_contents(dev, fused):
    """What a call handed out is not written again by later steps, compressions that leave a residual behind and ones that
    leave nothing among them; a tuple continued a second time does not touch what its first continuation returned."""
    from hqekv_amd.decode_layer import HqeAttentionLayer
    B, Hq, Hkv, D, T0, steps = 1, 8, 2, 128, 300, 72
    layer = HqeAttentionLayer(D, 0.2, 0.3, 0.5)
    layer.set_max_length(T0 + steps)
    layer.fused_step = fused
    data = [tuple(x.to(dev) for x in _qkv(B, Hq, Hkv, T0 if s == 0 else 1, D, 800 + s)) for s in range(steps + 1)]

    pkv, tuples = None, []
    for s in range(steps + 1):
        pkv = layer(*data[s], None, pkv)[2]
        tuples.append((pkv, tuple(x.to("cpu", copy=True) if torch.is_tensor(x) else x for x in pkv)))
    layer(*data[1], None, tuples[-2][0])
    for i, (kept, want) in enumerate(tuples):
        _same_tuple(kept, want, f"tuple {i}")


def test_a_step_over_classes_that_leave_positions_out_is_one_call_too(dev, monkeypatch):
    """Two tokens of a K class at one position, another position in none: ring row and appends ride in the attention call as
    they do over a whole cover, with the bits of the separate launches."""
    from hqekv_amd import _lib
    from hqekv_amd.decode_layer import HqeAttentionLayer
    B, Hq, Hkv, D, T0, steps = 2, 32, 8, 128, 350, 9
    data = [tuple(x.to(dev) for x in _qkv(B, Hq, Hkv, T0 if s == 0 else 1, D, 900 + s)) for s in range(steps + 1)]
    results, calls = [], []
    entry = _lib.load().hqekv_decode_step

    def counted(*a):
        calls.append(a)
        return entry(*a)
    monkeypatch.setattr(_lib.load(), "hqekv_decode_step", counted)
    for fused in (True, False):
        layer = HqeAttentionLayer(D, 0.2, 0.3, 0.5)
        layer.set_max_length(T0 + steps)
        layer.fused_step = fused
        pkv = list(layer(*data[0])[2])
        pkv[13] = pkv[13].clone()                    # positions of the 4-bit K class
        pkv[13][0] = pkv[13][1]
        pkv, outs = tuple(pkv), []
        for s in range(1, steps + 1):
            out, w, pkv, _ = layer(*data[s], None, pkv)
            outs += [out, w]
        results.append((outs, layer.last_weights.weights, pkv))
        assert len(calls) == steps                   # the first layer's, none of the second's
    for a, b in zip(results[0][0], results[1][0]):
        assert torch.equal(a, b)
    assert torch.equal(results[0][1], results[1][1])
    _same_tuple(results[0][2], tuple(x.cpu() if torch.is_tensor(x) else x for x in results[1][2]), "tuple")


@pytest.mark.parametrize("Hkv", [2, 1])
@pytest.mark.parametrize("kind", ["hqe", "kivi"])
def test_layers_take_projection_views(dev, kind, Hkv):
    """What a model hands over -- slices of one projection's (B, T, heads, D) output, seen per head -- gives the tuples and
    outputs of dense tensors, through prompt, compressions and steps."""
    from hqekv_amd.decode_layer import HqeAttentionLayer
    from hqekv_amd.kivi_layer import KiviAttentionLayer
    B, Hq, D, T0, steps = 2, 4 * Hkv, 128, 203, 40

    def run(views):
        if kind == "hqe":
            layer = HqeAttentionLayer(D, 0.2, 0.3, 0.5)
            layer.set_max_length(T0 + steps)
        else:
            layer = KiviAttentionLayer(D, 2, 2, 32, 32)
        pkv, outs = None, []
        for s in range(steps + 1):
            y = torch.cat(_qkv(B, Hq, Hkv, T0 if s == 0 else 1, D, 600 + s), 1).to(dev)
            if views:
                y = y.transpose(1, 2).contiguous().transpose(1, 2)
            parts = y[:, :Hq], y[:, Hq:Hq + Hkv], y[:, Hq + Hkv:]
            out, w, pkv = layer(*(parts if views else (x.contiguous() for x in parts)), None, pkv)[:3]
            outs += [out] + ([w] if w is not None else [])
        return outs, pkv
    (a, pa), (b, pb) = run(False), run(True)
    for x, y in zip(a, b):
        assert torch.equal(x, y)
    for i, (x, y) in enumerate(zip(pa, pb)):
        assert (x is None) == (y is None) and (not torch.is_tensor(x) or torch.equal(x, y)), i
